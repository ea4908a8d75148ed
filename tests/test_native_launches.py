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


P2, P3, P4, P5, P6, P7, STREAM = (P * k for k in range(2, 9))


def calls():
    """every launch with integer pointers, all arguments different: what the wrapper hands on"""
    gemm, body = R.make_desc(R.F16, 8, 8, 8, lda=3), R.make_elementwise_desc([("input", 0), ("input", 1), "add"], [(R.F32, 8, 1), (R.F32, 8, 1)], R.F32, 2, 8)
    att = R.make_attention_desc(R.F16, 1, 1, 256, 64, 96)
    return {"gemm": (gemm, P, P2, P3, P4, P5, P6, 77, STREAM), "fill": (R.F32, P, 2, 5, 4, 1.5, STREAM), "copy": (R.F32, P, 6, R.F16, P2, 9, 3, 7, STREAM),
            "reduce": (R.BF16, P, 4, 6, 5, 1, 3, 1, P2, P3, 78, STREAM), "elementwise": (body, [P, P2], None, STREAM), "softmax": (R.F16, P, 3, P2, 8, 2, 4, 2.5, P3, P4, 79, STREAM),
            "attention": (att, P, P2, P3, P4, P5, STREAM)}


@pytest.mark.parametrize("name", sorted(calls()))
def test_the_extension_carries_the_calls(name):
    """the library's status comes back through the extension (these are refused), not the None that sends a call by ctypes; what only ctypes takes is left to it"""
    f, args = getattr(R._bound(), name), calls()[name]
    status = f(*args)
    assert type(status) is int and status != 0, status
    assert f(*args[:-1], ctypes.c_void_p(STREAM)) is None and f(*args[:-1]) is None


def test_arguments_in_the_order_of_the_c_interface():
    """functions that note what they are called with, in the library's place"""
    native, L = R._bound(), R.lib()
    names = ("gemm", "fill", "copy", "reduce", "elementwise", "softmax", "attention")
    vp, i64, i32, size = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_size_t
    types = {"gemm": (vp,) * 7 + (size, vp), "fill": (i32, vp, i64, i64, i64, ctypes.c_double, vp), "copy": (i32, vp, i64, i32, vp, i64, i64, i64, vp),
             "reduce": (i32, vp, i64, i64, i64, i32, i32, i32, vp, vp, size, vp), "elementwise": (vp, ctypes.POINTER(vp), vp, vp),
             "softmax": (i32, vp, i64, vp, i64, i64, i64, ctypes.c_float, vp, vp, size, vp), "attention": (vp,) * 7}
    bind = lambda at: native.bind(R.GemmDesc, R.ElementwiseDesc, R.AttentionDesc, *at)
    seen = {}

    def stub(name):
        def record(*args):
            seen[name] = [tuple(a[:2]) if name == "elementwise" and i == 1 else a for i, a in enumerate(args)]
            return 40 + names.index(name)
        return ctypes.CFUNCTYPE(i32, *types[name])(record)
    stubs = [stub(n) for n in names]
    try:
        bind([ctypes.cast(s, vp).value for s in stubs])
        for i, name in enumerate(names):
            args = calls()[name]
            assert getattr(native, name)(*args) == 40 + i
            want = [ctypes.addressof(a) if isinstance(a, ctypes.Structure) else tuple(a) if isinstance(a, list) else a for a in args]
            assert seen[name] == want, name
    finally:
        bind([ctypes.cast(getattr(L, "frisk_hip_" + n), vp).value for n in names])
    assert "lda=3" in refused(R.gemm, R.make_desc(R.F16, 8, 8, 8, lda=3), P, P, P)
