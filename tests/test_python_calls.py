"""Runtime.call's native path: every kind of argument it converts reaches the entry point as ctypes would have passed it, and what it
does not convert (or a call that fails) takes the ctypes path."""
import ctypes as C
import gc
import os
import subprocess
import sys

import pytest

from sofie_amd import runtime as R

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class _Library:
    """The library, its contexts being rooms that no launch is made on: every call below ends before one."""

    def __init__(self):
        self.real, self.rooms, self.destroyed = R.load_library(), [], []

    def __getattr__(self, name):
        return getattr(self.real, name)

    def sofie_hip_ctx_create(self, out, device, stream):
        self.rooms.append(C.create_string_buffer(4096))
        out._obj.value = C.addressof(self.rooms[-1])
        return 0

    def sofie_hip_ctx_destroy(self, ctx):
        self.destroyed.append(ctx.value)
        return 0


@pytest.fixture
def library(monkeypatch):
    lib = _Library()
    monkeypatch.setattr(R, "load_library", lambda: lib)
    return lib


@pytest.fixture
def caller(library):
    rt = R.Runtime(0)
    return library, rt, rt.call


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
    _, rt, none = caller
    rt.ctx = None
    with pytest.raises(R.SofieHipError, match="NULL argument|ctx is NULL"):
        none("sofie_hip_gemm_f32", C.byref(R.GemmF32Desc()))


EMPTY = ("sofie_hip_fill_zero", 4096, 0)


def test_a_call_kept_past_close_is_refused(library):
    rt = R.Runtime(0)
    call = rt.call
    assert call(*EMPTY) is None
    rt.close()
    assert library.destroyed == [C.addressof(library.rooms[0])]
    for use in (call, rt.call):
        with pytest.raises(R.SofieHipError, match="ctx is NULL"):
            use(*EMPTY)


def test_a_call_that_is_kept_keeps_its_context(library):
    call = R.Runtime(0).call
    gc.collect()
    assert not library.destroyed and call(*EMPTY) is None
    del call
    gc.collect()
    assert len(library.destroyed) == 1


_D = R.GemmF32Desc()
POINTERS = [C.c_void_p(4096), C.c_void_p(), 4096, None, (C.c_float * 4)(), C.byref(_D), C.byref(_D, 8), _D, C.pointer(_D), C.c_void_p.from_param(5),
            C.c_int.from_param(5), C.c_int64.from_param(5), C.c_double.from_param(2.0), C.c_char_p.from_param(b"x"), C.c_char_p(b"x"), C.c_int(5), b"x", "x", 1.5]
INTEGERS = [0, 1, -1, True, 1 << 40, (1 << 63) + 5, 1.0, None, C.c_int32(1), C.c_int64(1), C.c_size_t(1), C.c_uint64(1), C.c_float(1), C.c_int.from_param(5), "1"]
REALS = [0.5, 0, True, C.c_float(0.5), C.c_double(0.5), C.c_int(1), C.c_float.from_param(0.5), None, "0.5"]


@pytest.mark.parametrize("name, before, kind, behind", [("sofie_hip_fill_zero", (), POINTERS, (0,)), ("sofie_hip_gemm_f32", (), POINTERS + [(R.GemmF32Desc * 2)(), C.byref(R.GemmI8Desc())], ()),
                                                        ("sofie_hip_softmax_f32", (None, None, 0, 4), INTEGERS, (0,)), ("sofie_hip_softmax_f32", (None, None, 0), INTEGERS, (1, 0)),
                                                        ("sofie_hip_fill_zero", (None,), INTEGERS, ()), ("sofie_hip_layernorm_f32", (None, None, None, None, 0, 8), REALS, (None, None))],
                         ids=["pointer", "structure", "int64", "int32", "size_t", "float"])
def test_what_ctypes_refuses_is_refused(caller, name, before, kind, behind):
    """Every kind of argument has the outcome of the plain ctypes call (which, as these calls do, ends before a launch)."""
    library, rt, call = caller

    def outcome(f):
        try:
            return f()
        except R.SofieHipError as e:
            return str(e)
        except Exception as e:
            return type(e)

    def plainly(*args):
        R._check(library, getattr(library, name)(rt.ctx, *args))
    for value in kind:
        args = before + (value,) + behind
        assert outcome(lambda: call(name, *args)) == outcome(lambda: plainly(*args)), value


def test_another_interpreter_calls_through_ctypes():
    """A build for one interpreter is none for another: the calls work, by the slower way."""
    assert R.load_library() and R._calls is not None
    code = """
import ctypes as C, importlib.machinery as machinery
machinery.EXTENSION_SUFFIXES[:] = [".another.so"]
from sofie_amd import runtime as R
rt = R.Runtime.__new__(R.Runtime)
rt.lib, room = R.load_library(), C.create_string_buffer(4096)
rt.ctx = C.c_void_p(C.addressof(room))
rt.call("sofie_hip_fill_zero", C.c_void_p(4096), 0)
try:
    rt.call("sofie_hip_gemm_f32", C.byref(R.GemmF32Desc()))
except R.SofieHipError as e:
    assert "batch" in str(e)
    print("refused")
rt.ctx = None
assert R._calls is None
"""
    assert subprocess.run([sys.executable, "-c", code], cwd=ROOT, stdout=subprocess.PIPE, check=True).stdout == b"refused\n"
