"""The float32-accuracy matrix-core kernels (csrc/split3.hip) at the sizes
where they can go wrong: single rows, the edges of the 32-row wave blocks and
128-row tiles, lengths that leave waves and workgroups empty, grouped heads,
partial tiles, both output dtypes; against the fp64 oracle under the parity
gate (tests/helpers.py; 1e-5 for float32).  Under that gate and tighter: the
float32 problems must be within 2e-6 of the oracle in norm (float32 sums of up
to a few hundred terms, three bfloat16 pieces per operand)."""
import numpy as np
import pytest

from tests.helpers import oracle, seeded_inputs
from tests.test_attention_gpu import run_case

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

CAUSAL = dict(is_causal=True)
HOLES = dict(mask_fn=lambda b, h, q, k: ((q + 3 * h - k) % 7 != 0) & (q // 40 != 2))


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("N", [1, 31, 33, 128, 129, 300])
def test_float32_causal_lengths(N, d):
    run_case((2, N, N, 2, 2, d), CAUSAL, "float32", scaled=False, seed=N)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_float32_gqa_partial_tiles_and_empty_rows(d):
    run_case((2, 257, 257, 4, 2, d), HOLES, "float32", scaled=False, seed=d)


@pytest.mark.parametrize("d", [64, 128])
def test_float32_cross_lengths(d):
    run_case((1, 70, 389, 4, 1, d), dict(block_size=64), "float32", scaled=False, seed=7)
    run_case((1, 389, 70, 2, 2, d), dict(block_size=64), "float32", scaled=False, seed=8)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("out", [None, "same"])
def test_wide_heads_16bit(dtype, out):
    od = dtype if out else None
    for N in (1, 33, 260):
        run_case((2, N, N, 2, 1, 256), CAUSAL, dtype, out_dtype=od, seed=N)
    run_case((1, 257, 257, 4, 2, 192), HOLES, dtype, out_dtype=od, seed=5)


@pytest.mark.parametrize("dtype,d", [("float32", 64), ("float32", 128), ("float32", 256), ("bfloat16", 256)])
def test_norm_relative_error(dtype, d):
    """O and the gradients of float32 accuracy: within 2e-6 of the float64 oracle
    in norm where they are stored in float32."""
    import jaxmodules_amd as jm

    B, N, H = 1, 384, 2
    Q, K, V, dO = seeded_inputs(B, N, N, H, H, d, 3, scaled=False)
    q, k, v = (torch.from_numpy(x).to("cuda", getattr(torch, dtype)).requires_grad_() for x in (Q, K, V))
    g = torch.from_numpy(dO).cuda()
    o = jm.masked_attention_via_map(q, k, v, is_causal=True)
    got = [o] + list(torch.autograd.grad(o, (q, k, v), g))
    O_ref, _, g_ref, _ = oracle(*(x.detach().float().cpu().numpy() for x in (q, k, v)), dO, CAUSAL)
    for name, a, b in zip(("O", "dQ", "dK", "dV"), got, [O_ref] + list(g_ref)):
        if a.dtype != torch.float32:
            continue
        a, b = a.detach().double().cpu().numpy(), np.asarray(b, np.float64)
        rel = np.linalg.norm(a - b) / np.linalg.norm(b)
        print(f"[norm] {dtype} d={d} {name}: {rel:.2e}")
        assert rel < 2e-6, name


@pytest.mark.parametrize("d", [64, 128, 256])
def test_large_logits(d):
    """Logits with a standard deviation of 10 (up to 50): a weight is off by its score's
    error times ln 2, so the scores' sums over d decide whether O meets the gate."""
    import jaxmodules_amd as jm
    from tests.helpers import assert_close

    for seed in range(3):
        Q, K, V, dO = seeded_inputs(1, 512, 512, 4, 2, d, seed, scaled=False)
        Q = (10 * Q).astype(np.float32)
        q, k, v = (torch.from_numpy(x).cuda() for x in (Q, K, V))
        o = jm.masked_attention_via_map(q, k, v, is_causal=True, precision="default")
        O_ref, _, _, _ = oracle(Q, K, V, dO, CAUSAL, grads=False)
        assert_close(o.cpu().numpy(), O_ref, "float32", f"d {d}")
