"""mattn_copy_rows (csrc/rows.hip): exact against torch's own padding, slicing and
conversion, over lengths with and without whole 16-byte chunks, strided and
heads-major rows, misaligned addresses, and several tensors of different sizes in one
launch; and the head dimensions that use it, end to end on such layouts."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

BF, F16, F32 = "bfloat16", "float16", "float32"


@pytest.mark.parametrize("src,dst", [(BF, BF), (F16, F16), (F32, F32), (BF, F32), (F16, F32), (F32, BF), (F32, F16)])
@pytest.mark.parametrize("sc,dc", [(80, 128), (128, 80), (37, 64), (64, 37), (1, 64), (40, 40), (256, 192)])
def test_copy_rows(src, dst, sc, dc):
    from jaxmodules_amd import attention as A

    gen = torch.Generator(device="cuda").manual_seed(sc + dc)
    pairs, want = [], []
    for n, (B, L, H) in enumerate(((2, 5, 3), (1, 33, 1), (3, 1, 7))):
        x = torch.randn((B, H, L, sc) if n == 1 else (B, L, H, sc), generator=gen, device="cuda").to(getattr(torch, src))
        if n == 1:
            x = x.transpose(1, 2)
        if n == 2:  # rows that start at odd addresses
            x = torch.randn((B, L, H, sc + 1), generator=gen, device="cuda").to(getattr(torch, src))[..., 1:]
        y = A._rows_like(x, dc, n == 1, getattr(torch, dst)).fill_(7.0)
        w = torch.zeros(y.shape, dtype=y.dtype, device="cuda")
        m = min(sc, dc)
        w[..., :m] = x[..., :m].to(y.dtype)
        pairs.append((x, y))
        want.append(w)
    A._copy_rows(pairs)
    for (_, y), w in zip(pairs, want):
        assert torch.equal(y, w)


@pytest.mark.parametrize("d", [20, 37, 96, 160])
def test_padded_head_dim_on_strided_inputs(d):
    """Q, K, V sliced out of one projection (odd d: rows at any alignment), 16-bit
    output and gradients equal to those of contiguous copies."""
    import jaxmodules_amd as jm

    gen = torch.Generator(device="cuda").manual_seed(d)
    qkv = torch.randn((2, 70, 3, 3 * d), generator=gen, device="cuda").to(torch.bfloat16)
    g = torch.randn((2, 3, 70, d), generator=gen, device="cuda").to(torch.bfloat16).transpose(1, 2)
    res = []
    for contiguous in (False, True):
        q, k, v = (x.contiguous() if contiguous else x for x in qkv.split(d, dim=-1))
        q, k, v = (x.detach().requires_grad_() for x in (q, k, v))
        o = jm.masked_attention_via_map(q, k, v, is_causal=True, out_dtype=torch.bfloat16)
        assert o.shape == (2, 70, 3, d) and o.dtype == torch.bfloat16
        res.append((o, *torch.autograd.grad(o, (q, k, v), g.contiguous() if contiguous else g)))
        with torch.no_grad():
            assert torch.equal(jm.masked_attention_via_map(q, k, v, is_causal=True, out_dtype=torch.bfloat16), o)
    for a, b in zip(*res):
        assert torch.equal(a, b)
