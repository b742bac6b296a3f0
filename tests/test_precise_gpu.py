"""precision="highest" on the float64 matrix cores (csrc/precise.hip) at the
sizes where it can go wrong: single rows, the edges of the 16-row wave blocks
and of the 64-row sub-blocks, grouped heads, partial tiles, empty rows, both
output dtypes, against the fp64 oracle under the parity gate (tests/helpers.py);
d = 300 keeps the D = 512 SIMT kernels covered."""
import pytest

from tests.test_attention_gpu import run_case

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

CAUSAL = dict(is_causal=True)
HOLES = dict(mask_fn=lambda b, h, q, k: ((q + 3 * h - k) % 7 != 0) & (q // 40 != 2))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_highest_lengths(dtype, d):
    for N in (1, 15, 17, 65, 129):
        run_case((2, N, N, 2, 2, d), CAUSAL, dtype, scaled=False, seed=N, precision="highest")


@pytest.mark.parametrize("dtype,out", [("float32", None), ("bfloat16", None), ("bfloat16", "bfloat16"),
                                       ("float16", "float16")])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_highest_gqa_partial_tiles_and_empty_rows(dtype, out, d):
    run_case((2, 257, 257, 4, 2, d), HOLES, dtype, out_dtype=out, seed=d, precision="highest")
    run_case((1, 70, 389, 4, 1, d), dict(block_size=64), dtype, out_dtype=out, seed=7, precision="highest")


@pytest.mark.parametrize("precision", [None, "highest"])
def test_d512(precision):
    run_case((1, 140, 140, 2, 1, 300), CAUSAL, "bfloat16", seed=2, precision=precision)
