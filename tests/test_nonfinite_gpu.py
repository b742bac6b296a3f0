"""Infinities, NaNs and the largest values in Q, K, V and dO on the float32-accuracy
matrix-core kernels (csrc/split3.hip): the results are those of the plain arithmetic over
the allowed pairs, in float64 here.  A masked pair adds nothing, whatever it holds."""
import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

INF = float("inf")
KINDS = [("float32", 64), ("float32", 128), ("float32", 256), ("bfloat16", 256), ("float16", 256)]


def _reference(q, k, v, do, allowed):
    """O, dQ, dK, dV as [N, H, d] sums over the allowed pairs alone."""
    q, k, v, do = (x.double() for x in (q, k, v, do))
    scale = 1 / math.sqrt(q.shape[-1])
    out = [torch.zeros_like(x) for x in (q, q, k, k)]
    for h in range(q.shape[1]):
        on = allowed[:, :, None]
        pair = lambda w, x: torch.where(on, w[:, :, None] * x, 0.0)  # noqa: E731  [N, L, d]
        s = torch.where(allowed, (q[:, None, h] * k[None, :, h]).sum(-1) * scale, -INF)
        m = torch.where(s.isnan(), -INF, s).amax(1, keepdim=True)
        p = torch.exp(s - torch.where(m == -INF, 0.0, m))
        p = torch.where(allowed, p / torch.where(allowed, p, 0.0).sum(1, keepdim=True), 0.0)
        o = pair(p, v[None, :, h]).sum(1)
        dp = (do[:, None, h] * (v[None, :, h] - o[:, None])).sum(-1)
        ds = p * dp * scale
        out[0][:, h] = o
        out[1][:, h] = pair(ds, k[None, :, h]).sum(1)
        out[2][:, h] = pair(ds, q[:, None, h]).sum(0)
        out[3][:, h] = pair(p, do[:, None, h]).sum(0)
    return out


@pytest.mark.parametrize("dtype,d", KINDS)
@pytest.mark.parametrize("what,value", [("v", INF), ("v", -INF), ("v", float("nan")), ("v", "largest"), ("k", INF),
                                        ("k", -INF), ("q", INF), ("do", INF)])
def test_values_that_are_not_finite(dtype, d, what, value):
    import jaxmodules_amd as jm

    N, H, dt = 150, 2, getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(d)
    t = {n: torch.randn((1, N, H, d), generator=gen, device="cuda").to(dt if n != "do" else torch.float32)
         for n in ("q", "k", "v", "do")}
    largest = value == "largest"  # (O alone: dO . V overflows)
    t[what][0, 70, 1, 5] = torch.finfo(dt).max if largest else value
    i = torch.arange(N, device="cuda")
    allowed = (i[:, None] >= i[None, :]) & ((i[:, None] + i[None, :]) % 3 != 0)
    q, k, v = (t[n].requires_grad_() for n in ("q", "k", "v"))
    o = jm.masked_attention_via_map(q, k, v, mask_fn=lambda b, h, q, k: (q >= k) & ((q + k) % 3 != 0))
    got = [o, *torch.autograd.grad(o, (q, k, v), t["do"])]
    want = _reference(*(t[n].detach()[0] for n in ("q", "k", "v", "do")), allowed)
    rel = 1e-5 if dtype == "float32" else 4e-3
    for name, a, b in list(zip(("O", "dQ", "dK", "dV"), got, want))[:1 if largest else 4]:
        a = a.detach()[0].double()
        assert torch.equal(a.isfinite(), b.isfinite()), name
        inf = b.isinf() & (name != "dV" or what == "do")  # (dV: a row that is NaN leaves Inf or NaN)
        assert torch.equal(a[inf], b[inf]), name
        fits = b.isfinite()
        assert ((a - b)[fits].norm() <= rel * b[fits].norm()).item(), name


@pytest.mark.parametrize("dtype,d", KINDS)
@pytest.mark.parametrize("what", ["q", "v", "do", "v and k", "q and k and v"])
def test_tensors_of_nan(dtype, d, what):
    """NaN wherever an allowed pair is, 0 in the rows and columns that have none (1 query in
    7, 1 key in 5), and a log-sum-exp that is right where only V is NaN: dV is finite."""
    import jaxmodules_amd as jm

    N, H, dt = 150, 2, getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(d + 1)
    t = {n: torch.randn((1, N, H, d), generator=gen, device="cuda").to(dt if n != "do" else torch.float32)
         for n in ("q", "k", "v", "do")}
    for n in what.split(" and "):
        t[n].fill_(float("nan"))
    if what == "v and k":  # (one key: the queries before it have finite scores)
        t["k"].nan_to_num_(1.0)[0, 70, 1, 5] = INF
    i = torch.arange(N, device="cuda")
    allowed = (i[:, None] >= i[None, :]) & (i[:, None] % 7 != 3) & (i[None, :] % 5 != 2)
    q, k, v = (t[n].requires_grad_() for n in ("q", "k", "v"))
    o = jm.masked_attention_via_map(q, k, v, mask_fn=lambda b, h, q, k: (q >= k) & (q % 7 != 3) & (k % 5 != 2))
    got = [o, *torch.autograd.grad(o, (q, k, v), t["do"])]
    want = _reference(*(t[n].detach()[0] for n in ("q", "k", "v", "do")), allowed)
    rel = 1e-5 if dtype == "float32" else 4e-3
    for name, a, b in zip(("O", "dQ", "dK", "dV"), got, want):
        a = a.detach()[0].double()
        fits = b.isfinite()
        assert torch.equal(a.isfinite(), fits), name
        assert ((a - b)[fits].norm() <= rel * b[fits].norm()).item(), name
