"""int8 and FP8 products of rows that start at any byte, which the kernels read as words: every phase of either operand's first byte, leading dimensions of every remainder, K and N
around whole steps, slabs and tiles, in each kernel that has such a reader, the operands with guard bytes of another value on both sides.  Whole numbers, exact in any order."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_tile_order import whole

pytestmark = pytest.mark.gpu
# M, N, K, bytes before A and B, bytes behind their rows
CASES = [(1, 16, 16, 1, 0, 0, 0), (5, 33, 129, 0, 3, 0, 0), (16, 65, 127, 2, 1, 1, 2), (33, 67, 256, 3, 2, 1, 3), (17, 129, 1025, 0, 0, 0, 2), (64, 64, 384, 1, 1, 0, 0),
         (130, 66, 257, 0, 2, 2, 1), (200, 71, 130, 3, 0, 0, 0), (40, 19, 2050, 2, 3, 0, 0), (129, 250, 47, 1, 2, 3, 3), (3, 40, 4227, 0, 0, 0, 0), (70, 131, 15, 1, 3, 0, 1)]


def placed(values, before, code):
    """The device copy of a matrix whose first byte lies `before` bytes behind a multiple of 16, guard bytes around it."""
    flat = np.full(values.size + before + 64, 0x55, dtype=np.uint8)
    flat[before : before + values.size] = code(values).reshape(-1)
    dev = util.to_dev(flat)
    return dev, C.c_void_p(dev.data_ptr() + before)


@pytest.mark.parametrize("tile", [0, 16, 32, 64, 164])
@pytest.mark.parametrize("transB", [0, 1])
@pytest.mark.parametrize("M,N,K,ba,bb,pa,pb", CASES)
def test_int8(rt, opt, M, N, K, ba, bb, pa, pb, transB, tile):
    a, b, bias = whole(5, (M, K + pa), 127), whole(6, (N, K + pb) if transB else (K, N + pb), 127), whole(7, (N,), 1000)
    code = lambda v: v.astype(np.int8).view(np.uint8)
    (dA, pA), (dB, pB) = placed(a, ba, code), placed(b, bb, code)
    dC, dY = util.to_dev(bias.astype(np.int32)), util.dev_empty((M, N), np.int32)
    g = R.GemmI8Desc()
    g.M, g.N, g.K, g.transB, g.lda, g.ldb, g.out, g.scale_scalar, g.q_scale = M, N, K, transB, K + pa, (K if transB else N) + pb, R.I8OUT_I32, 1.0, 1.0
    g.A, g.B, g.bias, g.Y = pA, pB, util.ptr(dC), util.ptr(dY)
    room = rt.lib.sofie_hip_gemm_i8_workspace(C.byref(g))
    ws = util.dev_empty((max(room, 256),), np.int8)
    g.workspace, g.workspace_bytes = util.ptr(ws), room
    torch.cuda.synchronize()
    opt("i8_tile", tile)
    rt.call("sofie_hip_gemm_i8", C.byref(g))
    rt.sync()
    assert np.array_equal(util.to_host(dY), a[:, :K] @ (b[:, :K].T if transB else b[:, :N]) + bias)


@pytest.mark.parametrize("tile", [0, 16, 32, 64, 164])
@pytest.mark.parametrize("M,N,K,ba,bb,pa,pb", CASES)
def test_fp8(rt, opt, M, N, K, ba, bb, pa, pb, tile):
    # |sum| <= 4227 * 64 < 2^24: exact in fp32
    a, b, bias = whole(8, (M, K), 8), whole(9, (N, K), 8), whole(10, (N,), 100)
    code = lambda v: torch.from_numpy(v.astype(np.float32)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    (dA, pA), (dB, pB) = placed(a, ba, code), placed(b, bb, code)
    dC, dY = util.to_dev(bias.astype(np.float32)), util.dev_empty((M, N), np.float32)
    g = R.GemmFp8Desc()
    g.M, g.N, g.K, g.transB, g.scale, g.act, g.out = M, N, K, 1, 1.0, R.ACT_NONE, R.F8OUT_F32
    g.A, g.B, g.bias, g.Y = pA, pB, util.ptr(dC), util.ptr(dY)
    torch.cuda.synchronize()
    opt("f8_tile", tile)
    rt.call("sofie_hip_gemm_fp8", C.byref(g))
    rt.sync()
    assert np.array_equal(util.to_host(dY), (a @ b.T + bias).astype(np.float32))


@pytest.mark.parametrize("tile", [0, 16, 32, 64, 164])
@pytest.mark.parametrize("M,N,K,ba,bb,pa,pb", CASES)
def test_fp8_columns(rt, opt, M, N, K, ba, bb, pa, pb, tile):
    """A B stored [K,N]: transposed on its way against rows read as words (as chosen, and by force in tiles of 128 x 64), or by a launch of its own (the other requests)."""
    a, b, bias = whole(30 + tile, (M, K + pa), 8), whole(31 + tile, (K, N + pb), 8), whole(32 + tile, (N,), 100)
    code = lambda v: torch.from_numpy(v.astype(np.float32)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    (dA, pA), (dB, pB) = placed(a, ba, code), placed(b, bb, code)
    dC, dY, ws = util.to_dev(bias.astype(np.float32)), util.dev_empty((M, N), np.float32), util.dev_empty(((N * K + 255) // 256 * 256,), np.int8)
    g = R.GemmFp8Desc()
    g.M, g.N, g.K, g.transB, g.lda, g.ldb, g.scale, g.act, g.out = M, N, K, 0, K + pa, N + pb, 1.0, R.ACT_NONE, R.F8OUT_F32
    g.A, g.B, g.bias, g.Y, g.workspace, g.workspace_bytes = pA, pB, util.ptr(dC), util.ptr(dY), util.ptr(ws), ws.numel()
    torch.cuda.synchronize()
    opt("f8_tile", tile)
    rt.call("sofie_hip_gemm_fp8", C.byref(g))
    rt.sync()
    assert np.array_equal(util.to_host(dY), (a[:, :K] @ b[:, :N] + bias).astype(np.float32))
