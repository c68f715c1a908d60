"""The general loop of int8 and FP8 products with tiles of 128 x 64, forced by the option: rows that start on any byte, a B stored [K,N] (which a thread transposes in pieces of four
columns there), K around a slab of 128 and shorter than one, tiles that are not filled.  Whole numbers, exact in any order."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_tile_order import whole

pytestmark = pytest.mark.gpu
SIZES = [(1, 16, 16), (128, 64, 128), (129, 65, 129), (127, 63, 127), (300, 200, 77), (131, 1000, 777), (260, 17, 1025), (64, 130, 383)]


@pytest.mark.parametrize("transB", [0, 1])
@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_int8(rt, opt, M, N, K, transB, pad):
    a, b, bias = whole(5, (M, K + pad), 127), whole(6, (N, K + pad) if transB else (K, N + pad), 127), whole(7, (N,), 1000)
    dA, dB, dC, dY = util.to_dev(a.astype(np.int8)), util.to_dev(b.astype(np.int8)), util.to_dev(bias.astype(np.int32)), util.dev_empty((M, N), np.int32)
    g = R.GemmI8Desc()
    g.M, g.N, g.K, g.transB, g.lda, g.ldb, g.out, g.scale_scalar, g.q_scale = M, N, K, transB, K + pad, (K if transB else N) + pad, R.I8OUT_I32, 1.0, 1.0
    g.A, g.B, g.bias, g.Y = util.ptr(dA), util.ptr(dB), util.ptr(dC), util.ptr(dY)
    room = rt.lib.sofie_hip_gemm_i8_workspace(C.byref(g))
    ws = util.dev_empty((max(room, 256),), np.int8)
    g.workspace, g.workspace_bytes = util.ptr(ws), room
    torch.cuda.synchronize()
    opt("i8_tile", 164)
    rt.call("sofie_hip_gemm_i8", C.byref(g))
    rt.sync()
    assert np.array_equal(util.to_host(dY), a[:, :K] @ (b[:, :K].T if transB else b[:, :N]) + bias)


@pytest.mark.parametrize("M,N,K", SIZES)
def test_fp8(rt, opt, M, N, K):
    a, b, bias = whole(8, (M, K), 8), whole(9, (N, K), 8), whole(10, (N,), 100)
    e4m3 = lambda v: util.to_dev(torch.from_numpy(v.astype(np.float32)).to(torch.float8_e4m3fn).view(torch.uint8).numpy())
    dA, dB, dC, dY = e4m3(a), e4m3(b), util.to_dev(bias.astype(np.float32)), util.dev_empty((M, N), np.float32)
    g = R.GemmFp8Desc()
    g.M, g.N, g.K, g.transB, g.scale, g.act, g.out = M, N, K, 1, 1.0, R.ACT_NONE, R.F8OUT_F32
    g.A, g.B, g.bias, g.Y = util.ptr(dA), util.ptr(dB), util.ptr(dC), util.ptr(dY)
    torch.cuda.synchronize()
    opt("f8_tile", 164)
    rt.call("sofie_hip_gemm_fp8", C.byref(g))
    rt.sync()
    assert np.array_equal(util.to_host(dY), (a @ b.T + bias).astype(np.float32))


@pytest.mark.parametrize("tile", [0, 164])
@pytest.mark.parametrize("pad_a, pad_b", [(0, 0), (3, 0), (4, 5)])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_fp8_columns(rt, opt, M, N, K, pad_a, pad_b, tile):
    """A B stored [K,N], by force in tiles of 128 x 64 and as chosen."""
    seed = 40 + tile + pad_a
    a, b, bias = whole(seed, (M, K + pad_a), 8), whole(seed + 1, (K, N + pad_b), 8), whole(seed + 2, (N,), 100)
    e4m3 = lambda v: util.to_dev(torch.from_numpy(v.astype(np.float32)).to(torch.float8_e4m3fn).view(torch.uint8).numpy())
    dA, dB, dC, dY = e4m3(a), e4m3(b), util.to_dev(bias.astype(np.float32)), util.dev_empty((M, N), np.float32)
    ws = util.dev_empty(((N * K + 255) // 256 * 256,), np.int8)
    g = R.GemmFp8Desc()
    g.M, g.N, g.K, g.transB, g.lda, g.ldb, g.scale, g.act, g.out = M, N, K, 0, K + pad_a, N + pad_b, 1.0, R.ACT_NONE, R.F8OUT_F32
    g.A, g.B, g.bias, g.Y, g.workspace, g.workspace_bytes = util.ptr(dA), util.ptr(dB), util.ptr(dC), util.ptr(dY), util.ptr(ws), ws.numel()
    torch.cuda.synchronize()
    opt("f8_tile", tile)
    rt.call("sofie_hip_gemm_fp8", C.byref(g))
    rt.sync()
    assert np.array_equal(util.to_host(dY), (a[:, :K] @ b[:, :N] + bias).astype(np.float32))
