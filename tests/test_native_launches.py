"""The calls of runtime.py that launch kernels: what the extension hands to the library, and what goes by ctypes as before.  Every call here is refused by the library before
anything touches a GPU, with a message that holds the arguments it looked at."""
import ctypes

import pytest

from frisk_amd import runtime as R

P = 0x1000


def refused(f, *args, **kw):
    with pytest.raises(R.FriskHipError) as e:
        f(*args, **kw)
    return str(e.value)


@pytest.mark.parametrize("p", [P, ctypes.c_void_p(P)], ids=["integer", "c_void_p"])
def test_arguments_arrive_in_their_places(p):
    bad = R.make_desc(R.F16, 8, 8, 8, lda=3)
    assert "lda=3 smaller than the stored row length 8" in refused(R.gemm, bad, p, p, p, None, None, None, 0, None)
    assert "leading dimension 4 smaller than the row length 5" in refused(R.fill, R.F32, p, 2, 5, 4, 1)
    assert "element type 77" in refused(R.fill, 77, p, 2, 5, 5, 1.5, p)
    assert "copy source: leading dimension 6 smaller than the row length 7" in refused(R.copy, R.F32, p, 6, R.F16, p, 9, 3, 7)
    assert "copy destination: leading dimension 6 smaller than the row length 7" in refused(R.copy, R.F32, p, 8, R.F16, p, 6, 3, 7, p)
    assert "copy destination: pointer is null" in refused(R.copy, R.F32, p, 8, R.F16, None, 8, 3, 7)
    assert "leading dimension 5 smaller than the row length 6" in refused(R.reduce, R.BF16, p, 4, 6, 5, 1, "max", True, p)
    assert refused(R.reduce, R.BF16, p, 4, 6, 6, 2, "max", True, p) and refused(R.reduce, R.BF16, p, 4, 6, 6, 0, 9, True, p) and refused(R.reduce, R.BF16, p, 4, 6, 6, 0, "add", True, None)
    assert "leading dimension 3 smaller than the row length 4" in refused(R.softmax, R.F16, p, 3, p, 8, 2, 4)
    assert "leading dimension 2 smaller than the row length 4" in refused(R.softmax, R.F16, p, 8, p, 2, 2, 4, 2, p, p, p, 16)
    assert refused(R.softmax, R.F16, p, 8, None, 8, 2, 4)
    body = R.make_elementwise_desc([("input", 0), ("input", 1), "add"], [(R.F32, 8, 1), (R.F32, 8, 1)], R.F32, 2, 8)
    for ins in ([p, None], (p, None), [p, 0]):
        assert "null" in refused(R.elementwise, body, ins, p)
    assert "null" in refused(R.elementwise, body, [p, p], None)
    assert refused(R.attention, R.make_attention_desc(R.F16, 1, 1, 256, 64, 96), p, p, p, p) and refused(R.attention, R.make_attention_desc(R.F16, 1, 1, 256, 64), p, None, p, p)


def test_what_the_extension_does_not_take_goes_by_ctypes():
    class Derived(R.GemmDesc):
        pass
    d = Derived.from_buffer_copy(bytes(R.make_desc(R.F16, 8, 8, 8, lda=3)))
    assert "lda=3" in refused(R.gemm, d, P, P, P)
    for f, args in ((R.gemm, (R.make_desc(R.F16, 8, 8, 8), 1.5, P, P)), (R.gemm, (R.make_attention_desc(R.F16, 1, 1, 256, 64), P, P, P)), (R.fill, (R.F32, P, "2", 5, 5, 1.0)),
                    (R.attention, (R.make_desc(R.F16, 8, 8, 8), P, P, P, P)), (R.copy, (R.F32, P, 6.0, R.F16, P, 9, 3, 7))):
        with pytest.raises((ctypes.ArgumentError, TypeError)):
            f(*args)
    with pytest.raises(TypeError):
        R.elementwise(R.make_elementwise_desc([("input", 0), "neg"], [(R.F32, 8, 1)], R.F32, 2, 8), ["x"], P)
