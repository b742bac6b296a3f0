"""Paths of the float32-accuracy and float64 matrix-core kernels (csrc/split3.hip,
csrc/precise.hip) that only large problems take: map rows and columns of more than 64
tiles (the walk's window of entries is refilled), more workgroups than the CUs take at
once (rounds of the launch order taken backwards, the last one partial), and row strides
that need 32 unsigned or 64 bits of offset.  Against float64 on the GPU."""
import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

F32, BF = torch.float32, torch.bfloat16


def _rand(shape, seed, dtype=F32):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _exact(q, k, v, do, allowed):
    """[O, dQ, dK, dV] of [1, L, H, d] tensors (Hq == Hkv), a head at a time."""
    out = [torch.empty(x.shape, dtype=torch.float64, device="cuda") for x in (q, q, k, k)]
    for h in range(q.shape[2]):
        a, b, c, g = (x[0, :, h].double() for x in (q, k, v, do))
        s = a @ b.T / math.sqrt(q.shape[3])
        p = torch.softmax(s if allowed is None else s.masked_fill_(~allowed, float("-inf")), 1)
        o = p @ c
        ds = p * (g @ c.T - (g * o).sum(1, keepdim=True)) / math.sqrt(q.shape[3])
        for x, y in zip(out, (o, ds @ b, ds.T @ a, p.T @ g)):
            x[0, :, h] = y
    return out


def _check(q, k, v, do, allowed=None, precision="default", **kw):
    import jaxmodules_amd as jm

    q, k, v = (x.requires_grad_() for x in (q, k, v))
    o = jm.masked_attention_via_map(q, k, v, precision=precision, out_dtype=do.dtype, **kw)
    got = (o, *torch.autograd.grad(o, (q, k, v), do))
    for name, a, b in zip(("O", "dQ", "dK", "dV"), got, _exact(*(x.detach() for x in (q, k, v, do)), allowed)):
        err = ((a.detach().double() - b).norm() / b.norm()).item()
        # float32 sums of up to 8500 terms in parts; 16-bit outputs: half a unit of 8 bits,
        # 2^-9 at most, 1.7e-3 in the mean
        print(f"[reach] {name}: {err:.1e}", flush=True)
        assert err < (2e-6 if a.dtype == F32 else 4e-3), name


@pytest.mark.parametrize("dtype,d", [(F32, 64), (F32, 128), (BF, 256)])
@pytest.mark.parametrize("Lq,Lk", [(40, 8500), (8500, 40), (300, 8230)])
def test_more_than_64_tiles(dtype, d, Lq, Lk):
    q, k, v = (_rand((1, n, 2, d), i, dtype) for i, n in enumerate((Lq, Lk, Lk)))
    do = _rand((1, Lq, 2, d), 3)
    _check(q, k, v, do, block_size=128)
    i, j = torch.arange(Lq, device="cuda")[:, None], torch.arange(Lk, device="cuda")[None]
    _check(q.detach(), k.detach(), v.detach(), do, (i + j) % 3 != 1, block_size=128,
           mask_fn=lambda b, h, q, k: (q + k) % 3 != 1)


@pytest.mark.parametrize("dtype,d,precision", [(F32, 64, "default"), (F32, 128, "default"), (BF, 256, "default"),
                                               (F32, 64, "highest"), (F32, 128, "highest")])
def test_more_workgroups_than_start_at_once(dtype, d, precision):
    """155 slots of a causal problem: 40 or 80 workgroups for each XCD's 32 CUs."""
    N, H = 31 * 128 - 50, 5
    q, k, v = (_rand((1, N, H, d), i, dtype) for i in range(3))
    i = torch.arange(N, device="cuda")
    _check(q, k, v, _rand((1, N, H, d), 3), i[:, None] >= i[None], precision, is_causal=True)


def _spread(x, stride):
    """x [1, N, 1, d] with `stride` elements between its rows."""
    N, d = x.shape[1], x.shape[3]
    y = torch.empty((N - 1) * stride + d, dtype=x.dtype, device="cuda").as_strided((1, N, 1, d), (d, stride, d, 1))
    return y.copy_(x)


@pytest.mark.parametrize("dtype,d,out", [(F32, 64, F32), (F32, 256, F32), (BF, 256, BF)])
def test_wide_stride_of_the_upstream_gradient(dtype, d, out):
    N = 40
    q, k, v = (_rand((1, N, 1, d), i, dtype) for i in range(3))
    _check(q, k, v, _spread(_rand((1, N, 1, d), 3, out), (1 << 24) + 8))


@pytest.mark.parametrize("precision", ["default", "highest"])
def test_wide_strides_of_the_inputs(precision):
    """64 rows of 12 million float32: offsets between 2^31 and 2^32 bytes."""
    N, d = 66, 64
    q, k, v = (_rand((1, N, 1, d), i) for i in range(3))
    _check(q, _spread(k, 12_000_000), _spread(v, 12_000_000), _rand((1, N, 1, d), 3), precision=precision)
