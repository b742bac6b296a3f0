"""Rows whose weight is all on one key, on the float32-accuracy matrix-core kernels
(csrc/split3.hip).  P = 1 and O = V there, so dP - delta = dO . (V - O) is what O's own
rounding leaves, and dQ and dK are that times scale K and scale Q: they must be, to
float32's (or the 16-bit outputs') relative accuracy.  Formed as the difference of two
float32 sums over d, dO . V and dO . O, it is those sums' rounding instead, 2 to 10
times as large and something else."""
import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
KINDS = [("float32", 64), ("float32", 128), ("float32", 256), ("bfloat16", 256), ("float16", 256)]


def _rand(shape, seed, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _check(q, k, v, do, key, **kw):
    """key [N]: the key each query's weight is on."""
    import jaxmodules_amd as jm

    half = q.dtype == torch.float16
    if half:  # gradients of 1e-7 times 2^7: float16's subnormals end at 6e-8
        do = do * 128
    q, k, v = (x.requires_grad_() for x in (q, k, v))
    o = jm.masked_attention_via_map(q, k, v, **kw)
    dq, dk, dv = (x.double() for x in torch.autograd.grad(o, (q, k, v), do))
    G, rel = q.shape[2] // k.shape[2], 1e-3 if q.dtype == torch.float32 else 4e-3
    q, k, v, o, do = (x.detach().double() for x in (q, k, v, o, do))
    kx, vx = (x.repeat_interleave(G, 2)[:, key] for x in (k, v))
    # P V over the sum of the weights: a few roundings of V at most
    assert ((o - vx).abs() <= 8 * U * vx.abs()).all()
    x = (do * (vx - o)).sum(-1, keepdim=True) / math.sqrt(q.shape[-1])
    per_key = lambda y: torch.zeros_like(k).index_add_(1, key, y.unflatten(2, (-1, G)).sum(3))  # noqa: E731
    for name, got, want in (("dQ", dq, x * kx), ("dK", dk, per_key(x * q)), ("dV", dv, per_key(do))):
        err, bound = (got - want).norm().item(), rel * want.norm().item()
        if name != "dV":  # the weights of the other keys, and a float16 output's subnormals
            bound += 1e-3 * U * ((do * vx).norm(dim=-1, keepdim=True) * {"dQ": kx, "dK": q}[name]).norm().item()
            bound += 2.0 ** -25 * got.numel() ** 0.5 if half else 0.0
        print(f"[dominated] d {q.shape[-1]} {name}: off by {err:.1e} of {want.norm().item():.1e}", flush=True)
        assert err <= bound, name


@pytest.mark.parametrize("dtype,d", KINDS)
def test_rows_with_one_key(dtype, d):
    from jaxmodules_amd import masks

    N, dt = 300, getattr(torch, dtype)
    q, k, v = (_rand((2, N, h, d), i, dt) for i, h in enumerate((4, 2, 2)))
    _check(q, k, v, _rand((2, N, 4, d), 3), torch.arange(N, device="cuda"), mask_fn=masks.window(0, 0))


@pytest.mark.parametrize("dtype,d", KINDS)
@pytest.mark.parametrize("sinks", [1, 5, 100])
def test_keys_that_queries_lean_on(dtype, d, sinks):
    """Every query has its weight on one of the first keys, at a logit of 60 (the others'
    weights are below e^-25, 2e-4 of u): up to all of them on one, more than the kernels
    keep a list of."""
    N, dt = 300, getattr(torch, dtype)
    k, v = _rand((1, N, 2, d), 1, dt), _rand((1, N, 2, d), 2, dt)
    key = torch.arange(N, device="cuda") % sinks
    kk = k[:, key].double()
    q = (kk / kk.pow(2).sum(-1, keepdim=True) * 60 * math.sqrt(d)).repeat_interleave(2, 2).to(dt)
    kt = k[0].double().repeat_interleave(2, 1).permute(1, 2, 0).contiguous()
    s = (q[0].double().transpose(0, 1).contiguous() @ kt) / math.sqrt(d)
    top = s.gather(2, key[None, :, None].expand(4, N, 1))
    s.scatter_(2, key[None, :, None].expand(4, N, 1), float("-inf"))
    assert (top - s.amax(2, keepdim=True)).min().item() > 25
    _check(q, k, v, _rand((1, N, 4, d), 3), key)
