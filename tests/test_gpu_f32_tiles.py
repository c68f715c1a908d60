"""Every kernel of the fp32 products and convolutions, forced by the context option "f32_tile", at sizes around the edges of its
tiles and slabs: one row or column more or less than a tile, reductions shorter than a slab, one k past a slab, and all four
storage orders with operands that allow 16-byte loads and operands that do not."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import binding as ob
from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_f32 import conv_desc, gemm

pytestmark = pytest.mark.gpu

TILES = [16, 32, 62, 64, 126, 128]


@pytest.fixture
def tile(rt, request):
    rt.set_option("f32_tile", request.param)
    yield request.param
    rt.set_option("f32_tile", 0)


@pytest.mark.parametrize("tile", TILES, indirect=True)
@pytest.mark.parametrize("transA,transB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (129, 65, 33), (127, 36, 31), (64, 128, 292), (132, 68, 16), (31, 260, 97)])
def test_products_around_tile_edges(rt, tile, M, N, K, transA, transB):
    A = util.normal(1, M * K).reshape((K, M) if transA else (M, K))
    B = util.normal(2, N * K, 0.05).reshape((N, K) if transB else (K, N))
    bias = util.normal(3, N)
    got = gemm(rt, A, B, bias, M, N, K, transA, transB, 1.25, 1.0, R.BIAS_ROW, R.ACT_LEAKYRELU, 0.1)
    a, b = (A.T if transA else A).astype(np.float64), (B.T if transB else B).astype(np.float64)
    want = 1.25 * (a @ b) + bias
    want = np.where(want >= 0, want, 0.1 * want)
    assert np.all(np.abs(got - want) <= 1e-5 * (1.25 * (np.abs(a) @ np.abs(b)) + 1.0))


@pytest.mark.parametrize("tile", TILES, indirect=True)
@pytest.mark.parametrize("case", [(2, 3, 9, 7, 5, 3, 3, (0, 0, 0, 0), (1, 1), (1, 1), 1), (3, 6, 13, 11, 70, 3, 2, (1, 0, 2, 1), (2, 1), (1, 2), 2),
                                  (1, 16, 16, 17, 33, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), 1), (2, 8, 12, 12, 130, 5, 5, (2, 2, 2, 2), (1, 1), (1, 1), 1)])
def test_convolutions_around_tile_edges(rt, tile, case):
    N, Cc, H, W, Cout, kh, kw, pads, strides, dils, group = case
    X = util.uniform01(30, N * Cc * H * W).reshape(N, Cc, H, W)
    Wt = util.normal(31, Cout * (Cc // group) * kh * kw, 0.3).reshape(Cout, Cc // group, kh, kw)
    b = util.normal(32, Cout)
    d = conv_desc(N, Cc, H, W, Cout, kh, kw, pads, strides, dils, group)
    dX, dW, db, dY = util.to_dev(X), util.to_dev(Wt), util.to_dev(b), util.dev_empty((N, Cout, d.OH, d.OW), np.float32)
    torch.cuda.synchronize()
    rt.call("sofie_hip_conv_f32", C.byref(d), util.ptr(dX), util.ptr(dW), util.ptr(db), R.ACT_RELU, C.c_float(0), util.ptr(dY), None, None)
    rt.sync()
    want = ob.conv_f32(X, Wt, b, pads=pads, strides=strides, dils=dils, group=group, act=1)
    assert np.abs(util.to_host(dY) - want).max() <= 1e-5 * max(1.0, float(np.abs(want).max()))


def conv2d_f64(X, Wt, pads):
    """Stride 1, one group; also the sum of the products' magnitudes, which bounds what rounding can do."""
    x = np.pad(X.astype(np.float64), ((0, 0), (0, 0), (pads[0], pads[2]), (pads[1], pads[3])))
    w = Wt.astype(np.float64).reshape(len(Wt), -1)
    windows = np.lib.stride_tricks.sliding_window_view(x, Wt.shape[2:], axis=(2, 3)).transpose(0, 2, 3, 1, 4, 5)
    columns = windows.reshape(*windows.shape[:3], -1)
    return [(c @ v.T).transpose(0, 3, 1, 2) for c, v in ((columns, w), (np.abs(columns), np.abs(w)))]


@pytest.mark.parametrize("tile", [0] + TILES, indirect=True)
@pytest.mark.parametrize("case", [(1, 1, 218, 219, 3, 216, 216, (0, 1, 1, 0)), (1, 3, 225, 224, 2, 224, 224, (0, 0, 0, 0)), (2, 1, 1, 50003, 4, 1, 50000, (0, 2, 0, 0)),
                                  (1, 2, 40000, 1, 5, 39998, 1, (0, 0, 0, 0))])
def test_convolutions_with_windows_of_any_length(rt, tile, case):
    """Reductions times window extents far beyond 2^31, which the index arithmetic of the gather has to divide exactly."""
    N, Cc, H, W, Cout, kh, kw, pads = case
    X = util.normal(33, N * Cc * H * W).reshape(N, Cc, H, W)
    Wt = util.normal(34, Cout * Cc * kh * kw, 0.1).reshape(Cout, Cc, kh, kw)
    d = conv_desc(N, Cc, H, W, Cout, kh, kw, pads, (1, 1), (1, 1), 1)
    dX, dW, dY = util.to_dev(X), util.to_dev(Wt), util.dev_empty((N, Cout, d.OH, d.OW), np.float32)
    torch.cuda.synchronize()
    print("conv", tile, case, flush=True)
    rt.call("sofie_hip_conv_f32", C.byref(d), util.ptr(dX), util.ptr(dW), None, R.ACT_NONE, C.c_float(0), util.ptr(dY), None, None)
    rt.sync()
    want, most = conv2d_f64(X, Wt, pads)
    assert np.all(np.abs(util.to_host(dY) - want) <= 1e-5 * most)
