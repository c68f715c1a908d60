"""Which tile a workgroup takes (TileOrder of mfma8_common.hpp): every tile of every product of a batch exactly once, at tile counts around the eight XCDs, the bands and the last band, in
every order that the option "swizzle" names.  Results are whole numbers, which every kernel gives exactly."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu


def whole(seed, shape, most):
    return (util.uniform01(seed, int(np.prod(shape))) * (2 * most + 1)).astype(np.int64).reshape(shape) - most


@pytest.mark.parametrize("tile", [16, 32, 64])
@pytest.mark.parametrize("batch", [1, 2, 7, 8, 9, 33])
@pytest.mark.parametrize("tiles_m, tiles_n", [(1, 1), (1, 9), (4, 2), (5, 3), (9, 1), (7, 5)])
def test_products_of_a_batch(rt, opt, tile, batch, tiles_m, tiles_n):
    M, N, K = tiles_m * tile - 3, tiles_n * tile - 1, 20
    a, b = whole(1, (batch, M, K), 8), whole(2, (batch, N, K), 8)
    dA, dB, dY = util.to_dev(a.astype(np.float32)), util.to_dev(b.astype(np.float32)), util.dev_empty((batch, M, N), np.float32)
    g = R.GemmF32Desc()
    g.M, g.N, g.K, g.transB, g.alpha, g.batch = M, N, K, 1, 1.0, batch
    g.A, g.B, g.Y = util.ptr(dA), util.ptr(dB), util.ptr(dY)
    g.strideA, g.strideB, g.strideY = M * K, N * K, M * N
    torch.cuda.synchronize()
    opt("f32_tile", tile)
    rt.call("sofie_hip_gemm_f32", C.byref(g))
    rt.sync()
    assert np.array_equal(util.to_host(dY), a @ b.transpose(0, 2, 1))


@pytest.mark.parametrize("swizzle", [0, 1, 3, 4, 255, 0x100, 0x104])
@pytest.mark.parametrize("tile", [16, 64])
@pytest.mark.parametrize("tiles_m, tiles_n", [(1, 1), (3, 17), (5, 3), (8, 8), (13, 1)])
def test_orders(rt, opt, swizzle, tile, tiles_m, tiles_n):
    M, N, K = tiles_m * tile, tiles_n * tile, 64
    a, b = whole(3, (M, K), 127), whole(4, (N, K), 127)
    dA, dB, dY = util.to_dev(a.astype(np.int8)), util.to_dev(b.astype(np.int8)), util.dev_empty((M, N), np.int32)
    g = R.GemmI8Desc()
    g.M, g.N, g.K, g.transB, g.out, g.scale_scalar, g.q_scale = M, N, K, 1, R.I8OUT_I32, 1.0, 1.0
    g.A, g.B, g.Y = util.ptr(dA), util.ptr(dB), util.ptr(dY)
    torch.cuda.synchronize()
    opt("swizzle", swizzle)
    opt("i8_tile", tile)
    rt.call("sofie_hip_gemm_i8", C.byref(g))
    rt.sync()
    assert np.array_equal(util.to_host(dY), a @ b.T)
