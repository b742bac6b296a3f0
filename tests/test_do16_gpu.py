"""A 16-bit dO read as it is (MATTN_DO_16) gives the gradients of the same dO in
float32: bitwise for the matrix products' operands (both are exact copies), up to the
summation order of delta = rowsum(dO * O)."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("d", [64, 80, 128, 256])
@pytest.mark.parametrize("N", [1, 130, 384])
def test_16bit_upstream_gradient(dtype, d, N):
    import jaxmodules_amd as jm

    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(N + d)
    q, k, v, g = (torch.randn((2, N, 4, d), generator=gen, device="cuda").to(dt) for _ in range(4))
    q, k, v = (x.requires_grad_() for x in (q, k, v))
    res = []
    for out in (dt, torch.float32):
        o = jm.masked_attention_via_map(q, k, v, is_causal=True, out_dtype=out)
        res.append(torch.autograd.grad(o, (q, k, v), g.to(out)))
    # delta is a sum of d terms dO O in another order: off by at most 2 d 2^-24 of the
    # terms' magnitudes (|O| <= max |V|), which dS carries times P: P sums to 1 over a
    # row's keys (dQ) and to at most N over a key's rows (dK), and each side is then
    # rounded to its 16-bit type
    w = 2 * d * 2.0 ** -24 * (g.abs().sum(-1).max() * v.abs().max()).item() * d ** -0.5
    eps = 2.0 ** (-8 if dtype == "bfloat16" else -11)
    for name, a, b, t in zip(("dQ", "dK", "dV"), *res, (w * k.abs().max().item(), w * N * q.abs().max().item(), 0.0)):
        if name == "dV":  # no delta in it
            assert torch.equal(a, b)
        a, b = a.double(), b.double()
        assert ((a - b).abs() <= t + eps * b.abs() + 2.0 ** -24).all(), name
        if N > 1:
            assert (a != b).double().mean() < 0.02, name


@pytest.mark.parametrize("d", [64, 80, 256])
def test_16bit_upstream_gradient_at_an_odd_address(d):
    """The gradient of a slice of a flat buffer: dense, but not at a 16-byte address; and
    one expanded over the sequence.  Bitwise the gradients of an ordinary copy."""
    import jaxmodules_amd as jm

    gen = torch.Generator(device="cuda").manual_seed(d)
    q, k, v = (torch.randn((1, 130, 2, d), generator=gen, device="cuda").to(torch.bfloat16).requires_grad_()
               for _ in range(3))
    flat = torch.randn(130 * 2 * d + 1, generator=gen, device="cuda").to(torch.bfloat16)
    for g in (flat[1:].view(1, 130, 2, d), flat[:2 * d].view(1, 1, 2, d).expand(1, 130, 2, d)):
        o = jm.masked_attention_via_map(q, k, v, is_causal=True, out_dtype=torch.bfloat16)
        got = torch.autograd.grad(o, (q, k, v), g, retain_graph=True)
        want = torch.autograd.grad(o, (q, k, v), g.clone(memory_format=torch.contiguous_format))
        for a, b in zip(got, want):
            assert torch.equal(a, b)


def test_flag_is_refused_where_no_kernel_takes_it():
    from jaxmodules_amd import _lib
    from tests.test_capi import _problem

    import ctypes

    lib = _lib.load()
    check = lambda **kw: lib.mattn_validate(ctypes.byref(_problem(flags=_lib.MATTN_DO_16, **kw)), None)  # noqa: E731
    assert check() == 0 and check(D=256) == 0
    assert check(dtype=_lib.MATTN_F32, o_dtype=_lib.MATTN_F32) == -4
    assert check(D=512) == -4
    p = _problem(flags=_lib.MATTN_DO_16 | _lib.MATTN_PRECISE)
    assert lib.mattn_validate(ctypes.byref(p), None) == -4
