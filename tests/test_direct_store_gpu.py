"""A 16-bit O that the kernels round themselves (no gradient needed) holds the bits of the
one that is rounded from their float32 O (training): every kernel family, over padded head
dimensions, ragged lengths, empty rows, split rows, heads-major and strided outputs."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _rand(shape, seed, dtype, scale=1.0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=gen, device="cuda") * scale).to(dtype)


def _check(fn, q, k, v, **kw):
    q, k, v = (x.requires_grad_() for x in (q, k, v))
    o = fn(q, k, v, out_dtype=q.dtype, **kw)
    assert o.requires_grad and o.dtype == q.dtype
    direct = fn(q.detach(), k.detach(), v.detach(), out_dtype=q.dtype, **kw)
    assert not direct.requires_grad and torch.equal(direct, o)
    with torch.no_grad():
        off = fn(q, k, v, out_dtype=q.dtype, **kw)
    assert not off.requires_grad and torch.equal(off, o)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 80, 128, 256])
@pytest.mark.parametrize("precision", ["default", "highest"])
def test_same_bits(dtype, d, precision):
    import jaxmodules_amd as jm

    run = jm.masked_attention_via_map
    holes = lambda b, h, q, k: ((q + 3 * h - k) % 7 != 0) & (q // 40 != 2)  # noqa: E731
    for N, L, H, Hkv, scale, kw in (
            (130, 130, 4, 2, d ** -0.25, dict(is_causal=True)),
            (257, 257, 2, 2, 1.0, dict(mask_fn=holes)),          # empty rows
            (300, 300, 2, 1, 4.0, dict(is_causal=True)),         # sharp rows
            (70, 389, 2, 2, 1.0, dict(block_size=64))):
        q, k, v = _rand((2, N, H, d), N, dtype, scale), _rand((2, L, Hkv, d), 1, dtype, scale), _rand((2, L, Hkv, d), 2, dtype)
        _check(run, q, k, v, precision=precision, **kw)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 96, 256])
def test_same_bits_heads_major(dtype, d):
    import jaxmodules_amd as jm

    q, k, v = _rand((2, 4, 256, d), 0, dtype, 2.0), _rand((2, 2, 256, d), 1, dtype), _rand((2, 2, 256, d), 2, dtype)
    _check(jm.flex_attention, q, k, v, block_mask=jm.BlockMask.causal_mask(1, 1, 256, 256, 128), enable_gqa=True)


@pytest.mark.parametrize("d", [64, 80])
def test_same_bits_strided(d):
    import jaxmodules_amd as jm
    from jaxmodules_amd import masks

    mask = masks.intersect(masks.same_residue(16), masks.causal())
    q, k, v = (_rand((1, 2048, 2, d), i, torch.float16) for i in range(3))
    _check(jm.masked_attention_via_map, q, k, v, mask_fn=mask)


def test_no_grad_writes_no_float32_output():
    """Under no_grad a call on inputs that require a gradient keeps nothing for it."""
    import jaxmodules_amd as jm

    q, k, v = (_rand((1, 4096, 8, 128), i, torch.bfloat16).requires_grad_() for i in range(3))
    run = lambda *t: jm.masked_attention_via_map(*t, is_causal=True, out_dtype=torch.bfloat16)  # noqa: E731
    peaks = []
    for t in ((q.detach(), k.detach(), v.detach()), (q, k, v)):
        run(*t)
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        with torch.no_grad():
            run(*t)
        peaks.append(torch.cuda.max_memory_allocated() - base)
    assert peaks[1] == peaks[0], peaks
