"""Runtime.call's native path: every kind of argument it converts reaches the entry point as ctypes would have passed it, and what it
does not convert (or a call that fails) takes the ctypes path."""
import ctypes as C

import pytest

from sofie_amd import runtime as R


@pytest.fixture(scope="module")
def caller():
    lib = R.load_library()
    room = C.create_string_buffer(4096)          # a context that no launch is made on: every call below ends before one
    return lib, room, R._calls.caller(C.addressof(room), R._call_slowly)


@pytest.mark.parametrize("pointer", [C.c_void_p(4096), 4096, (C.c_float * 4)(), C.byref(C.c_float())], ids=["c_void_p", "int", "array", "byref"])
def test_empty_calls_are_taken(caller, pointer):
    _, _, call = caller
    assert call("sofie_hip_softmax_f32", pointer, pointer, 0, 10, 1, 0) is None
    assert call("sofie_hip_transpose_i8", pointer, pointer, 0, 10, 0, 0) is None
    assert call("sofie_hip_fill_zero", pointer, C.c_size_t(0)) is None
    assert call("sofie_hip_layernorm_f32", pointer, pointer, pointer, pointer, 0, 8, C.c_float(1e-5), None, None) is None
    assert call("sofie_hip_layernorm_f32", pointer, pointer, pointer, pointer, 0, 8, 1e-5, None, None) is None


def test_fields_arrive(caller):
    """The message of a refused call names what the entry point read."""
    _, _, call = caller
    d = (R.GemmF32Desc * 2)()
    d[1].batch, d[1].M, d[1].N = 1, -3, 5
    with pytest.raises(R.SofieHipError, match="batch must be >= 1"):
        call("sofie_hip_gemm_f32", C.byref(d[0]))
    with pytest.raises(R.SofieHipError, match="negative"):
        call("sofie_hip_gemm_f32", C.byref(d[1]))
    with pytest.raises(R.SofieHipError, match="q_scale"):
        g = R.GemmI8Desc()
        g.M = g.N = 1
        g.Y, g.out = 4096, R.I8OUT_I8_DQQ
        call("sofie_hip_gemm_i8", C.byref(g))
    with pytest.raises(R.SofieHipError, match="negative shape"):
        call("sofie_hip_transpose_i8", 4096, 4096, -1, 10, 0, 0)


def test_wrong_arguments_raise(caller):
    _, _, call = caller
    with pytest.raises(C.ArgumentError):
        call("sofie_hip_gemm_f32", C.byref(R.GemmI8Desc()))     # another structure
    with pytest.raises(TypeError):
        call("sofie_hip_gemm_f32")
    with pytest.raises(C.ArgumentError):
        call("sofie_hip_fill_zero", 4096, "eight")
    with pytest.raises(AttributeError):
        call("sofie_hip_no_such_entry", 1)


def test_no_context(caller):
    none = R._calls.caller(0, R._call_slowly)
    with pytest.raises(R.SofieHipError, match="NULL argument|ctx is NULL"):
        none("sofie_hip_gemm_f32", C.byref(R.GemmF32Desc()))
