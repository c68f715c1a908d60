"""The int8 / FP8 kernels for few rows (direct: tiles of 16 x 16 and 32 x 32, waves that split the reduction) and for rows of any
length and alignment (general loop, B stored either way) at the edges of their tiles, steps and slabs: one row, one column, K
shorter than a chunk, one byte past a chunk, a step and a slab, operands that start at odd addresses."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import binding as ob
from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_gemm_i8 import run_gemm

pytestmark = pytest.mark.gpu


@pytest.fixture
def tile(rt, request):
    for name in ("i8_tile", "f8_tile"):
        rt.set_option(name, request.param)
    yield request.param
    for name in ("i8_tile", "f8_tile"):
        rt.set_option(name, 0)


SHAPES = [(1, 1, 1), (5, 3, 15), (16, 16, 16), (17, 33, 127), (15, 31, 129), (65, 66, 145), (130, 129, 257), (33, 260, 1000)]


@pytest.mark.parametrize("tile", [0, 16, 32, 64, 128], indirect=True)
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("transB", [0, 1])
def test_int8_products(rt, tile, M, N, K, transB):
    A = util.int8_sym(1, M * K).reshape(M, K)
    B = util.int8_sym(2, N * K).reshape((N, K) if transB else (K, N))
    bias = util.int32_range(3, N, -5000, 5000)
    scale = ((0.5 + util.uniform01(4, N)) / np.float32(60.0 * np.sqrt(K))).astype(np.float32)
    acc = A.astype(np.int64) @ (B.T if transB else B).astype(np.int64)
    assert np.array_equal(run_gemm(rt, A, B, M, N, K, transB=transB, out=R.I8OUT_I32), acc)
    got = run_gemm(rt, A, B, M, N, K, transB=transB, out=R.I8OUT_I8, bias=bias, scale=scale, relu_out=1)
    want = np.clip(np.rint((acc + bias).astype(np.float32) * scale), -128, 127)
    assert np.array_equal(got, np.maximum(want, 0).astype(np.int8))


@pytest.mark.parametrize("shift", [1, 3, 8])
@pytest.mark.parametrize("transB", [0, 1])
@pytest.mark.parametrize("M,N,K", [(7, 20, 200), (70, 100, 333), (300, 200, 128)])
def test_operands_that_start_at_odd_addresses(rt, M, N, K, transB, shift):
    A = util.int8_sym(5, M * K).reshape(M, K)
    B = util.int8_sym(6, N * K).reshape((N, K) if transB else (K, N))
    dA, dB = util.dev_empty((M * K + shift,), np.int8), util.dev_empty((N * K + shift,), np.int8)
    dA[shift:].copy_(util.to_dev(A.reshape(-1)))
    dB[shift:].copy_(util.to_dev(B.reshape(-1)))
    dY = util.dev_empty((M, N), np.int32)
    d = R.GemmI8Desc()
    d.M, d.N, d.K, d.transB, d.out = M, N, K, transB, R.I8OUT_I32
    d.A, d.B, d.Y = C.c_void_p(dA.data_ptr() + shift), C.c_void_p(dB.data_ptr() + shift), util.ptr(dY)
    d.scale_scalar = d.q_scale = 1.0
    need = rt.lib.sofie_hip_gemm_i8_workspace(C.byref(d))
    ws = util.dev_empty((max(need, 256),), np.int8)
    d.workspace, d.workspace_bytes = util.ptr(ws), need
    torch.cuda.synchronize()
    rt.call("sofie_hip_gemm_i8", C.byref(d))
    rt.sync()
    assert np.array_equal(util.to_host(dY), A.astype(np.int64) @ (B.T if transB else B).astype(np.int64))


@pytest.mark.parametrize("tile", [0, 16, 32, 64, 128], indirect=True)
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("transB", [0, 1])
def test_fp8_products(rt, tile, M, N, K, transB):
    A = ob.quantize_fp8(util.normal(7, M * K).reshape(M, K), 1.0)
    B = ob.quantize_fp8(util.normal(8, N * K).reshape((N, K) if transB else (K, N)), 1.0)
    dA, dB, dY = util.to_dev(A), util.to_dev(B), util.dev_empty((M, N), np.float32)
    ws = util.dev_empty((K * N + 256,), np.uint8)
    d = R.GemmFp8Desc()
    d.M, d.N, d.K, d.transB, d.scale, d.out = M, N, K, transB, 0.5, R.F8OUT_F32
    d.A, d.B, d.Y, d.workspace, d.workspace_bytes = util.ptr(dA), util.ptr(dB), util.ptr(dY), util.ptr(ws), K * N + 256
    torch.cuda.synchronize()
    rt.call("sofie_hip_gemm_fp8", C.byref(d))
    rt.sync()
    a, b = ob.e4m3_to_f32(A).astype(np.float64), ob.e4m3_to_f32(B).astype(np.float64)
    b = b.T if transB else b
    want = 0.5 * (a @ b)
    assert np.all(np.abs(util.to_host(dY) - want) <= 2.0 ** -14 * 0.5 * (np.abs(a) @ np.abs(b)) + 1e-6 * np.abs(want) + 1e-12)
