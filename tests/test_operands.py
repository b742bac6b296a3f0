"""What the kernels are handed: rows at 16-byte addresses with 16-byte strides
(attention._ready), on the CPU."""
import pytest

torch = pytest.importorskip("torch")

from jaxmodules_amd import attention as A


def _views():
    flat = torch.arange(4 * 6 * 2 * 64 + 8, dtype=torch.float32).to(torch.bfloat16)
    n = 4 * 6 * 2 * 64
    dense = flat[:n].view(4, 6, 2, 64)
    yield "aligned", dense, True
    yield "strided rows", dense.transpose(0, 1), True
    yield "expanded over the sequence", dense[:, :1].expand(4, 6, 2, 64), True
    yield "dense at an odd address", flat[1:n + 1].view(4, 6, 2, 64), False
    yield "odd stride on a dimension of one", flat[:n].as_strided((1, 6, 2, 64), (n + 3, 128, 64, 1)), False
    yield "d not contiguous", flat[:n].view(4, 6, 64, 2).transpose(2, 3), False


@pytest.mark.parametrize("what,x,as_is", list(_views()), ids=lambda v: v if isinstance(v, str) else "")
def test_ready(what, x, as_is):
    y = A._ready(x)
    assert (y is x) == as_is
    assert torch.equal(x, y) and y.dtype == x.dtype
    assert y.data_ptr() % 16 == 0 and y.stride(3) == 1
    assert all(s * y.element_size() % 16 == 0 for s in y.stride()[:3])


@pytest.mark.parametrize("q,o,do", [("float16", "float32", "bfloat16"), ("float16", "float16", "float32"),
                                    ("bfloat16", "bfloat16", "float16"), ("float32", "float32", "bfloat16")])
def test_upstream_gradient_of_another_dtype_is_refused(q, o, do):
    """A dO that is neither of O's dtype nor of the inputs' beside a float32 O would be
    read as something else."""
    from types import SimpleNamespace

    t = [torch.zeros((1, 128, 1, 64), dtype=getattr(torch, n)) for n in (q, o, do)]
    tm = SimpleNamespace(B=1, Lq=128, Hq=1, Lk=128, Hkv=1)
    with pytest.raises(TypeError, match="dO must have"):
        A.mattn_backward(t[0], t[0], t[0], t[1], torch.zeros(1, 1, 128), t[2], tm, 0.125)


def test_scale_past_float32_is_the_library_s_to_refuse():
    import ctypes

    from jaxmodules_amd import _lib

    q = torch.zeros((1, 128, 1, 64))
    p = A._problem(q, q, q, q, 1e39)
    assert p.scale == float("inf")
    assert _lib.load().mattn_validate(ctypes.byref(p), None) == -2  # MATTN_ERR_SHAPE
    assert A._problem(q, q, q, q, 3e38).scale > 2.9e38
