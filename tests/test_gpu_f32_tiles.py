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


def with_nonfinite(a, seed):
    """Some elements, the last among them, replaced by infinities of both signs, a NaN, both zeros and a large number."""
    a = a.copy()
    at = (util.uniform01(seed, 12) * a.size).astype(int)
    a.reshape(-1)[at] = [np.inf, -np.inf, np.nan, 0.0, -0.0, 1.0e30] * 2
    a.reshape(-1)[-1] = np.inf
    return a


def same_as_ieee(got, want, most):
    """NaN and infinities where the sums of IEEE products have them, everything else within rounding."""
    assert np.array_equal(np.isnan(got), np.isnan(want))
    infinite = np.isinf(want)
    assert np.array_equal(got[infinite], want[infinite].astype(np.float32)) and (infinite.any() or np.isnan(want).any())
    rest = np.isfinite(want)
    assert rest.any() and np.all(np.abs(got[rest] - want[rest]) <= 1e-5 * most[rest])


@pytest.mark.parametrize("tile", [0] + TILES, indirect=True)
@pytest.mark.parametrize("transA,transB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(132, 68, 52), (35, 130, 33)])
def test_products_of_nan_and_infinity(rt, tile, M, N, K, transA, transB):
    """What pads a tile or a slab is zero on both sides: a NaN or an infinity reaches its own row and column only."""
    A = with_nonfinite(util.normal(50, M * K), 51).reshape((K, M) if transA else (M, K))
    B = util.normal(52, N * K).reshape((K, N) if transB == 0 else (N, K))
    B.reshape(-1)[::97] = 0.0                              # infinity times zero
    B.reshape(-1)[-1] = -np.inf
    got = gemm(rt, A, B, None, M, N, K, transA, transB)
    a, b = (A.T if transA else A).astype(np.float64), (B.T if transB else B).astype(np.float64)
    with np.errstate(invalid="ignore"):
        products = a[:, None, :] * b.T[None, :, :]
        want, most = products.sum(2), np.abs(products).sum(2)
    same_as_ieee(got, want, most)


@pytest.mark.parametrize("tile", [0, 3032, 3064, 3128] + TILES, indirect=True)
@pytest.mark.parametrize("case", [(2, 9, 13, 11, 35, 3), (2, 2, 9, 10, 33, 2), (1, 3, 40, 41, 5, 6)])
def test_convolutions_of_nan_and_infinity(rt, tile, case):
    """The same for the padding of an image, which is a zero (times an infinite weight: a NaN, as in the reference's column matrix)."""
    N, Cc, H, W, Cout, k = case
    X = with_nonfinite(util.normal(53, N * Cc * H * W), 54).reshape(N, Cc, H, W)
    Wt = util.normal(55, Cout * Cc * k * k).reshape(Cout, Cc, k, k)
    Wt[1, 0, 0, 0] = np.inf
    d = conv_desc(N, Cc, H, W, Cout, k, k, (1, 1, 1, 1), (1, 1), (1, 1), 1)
    dX, dW, dY = util.to_dev(X), util.to_dev(Wt), util.dev_empty((N, Cout, d.OH, d.OW), np.float32)
    torch.cuda.synchronize()
    rt.call("sofie_hip_conv_f32", C.byref(d), util.ptr(dX), util.ptr(dW), None, R.ACT_NONE, C.c_float(0), util.ptr(dY), None, None)
    rt.sync()
    x = np.pad(X.astype(np.float64), ((0, 0), (0, 0), (1, 1), (1, 1)))
    windows = np.lib.stride_tricks.sliding_window_view(x, (k, k), axis=(2, 3)).transpose(0, 2, 3, 1, 4, 5).reshape(N, 1, d.OH, d.OW, -1)
    with np.errstate(invalid="ignore"):
        products = windows * Wt.astype(np.float64).reshape(1, Cout, 1, 1, -1)
        same_as_ieee(util.to_host(dY), products.sum(4), np.abs(products).sum(4))


@pytest.mark.parametrize("tile", [0] + TILES, indirect=True)
@pytest.mark.parametrize("transA,transB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K,gap", [(66, 36, 40, 4), (66, 36, 40, 8), (33, 35, 31, 3), (64, 64, 32, 1)])
def test_batched_products_with_padded_pitches(rt, tile, M, N, K, gap, transA, transB):
    """Rows `gap` floats longer than the matrix and matrices some rows apart: the gaps hold NaN, are not read and not written."""
    batch = 3
    rows_a, cols_a, rows_b, cols_b = (K, M, N, K) if transA and transB else (K, M, K, N) if transA else (M, K, N, K) if transB else (M, K, K, N)

    def padded(seed, rows, cols, scale=1.0):
        whole = np.full((batch, rows + 2, cols + gap), np.nan, np.float32)
        whole[:, :rows, :cols] = util.normal(seed, batch * rows * cols, scale).reshape(batch, rows, cols)
        return whole, whole[:, :rows, :cols]
    (wa, a), (wb, b), (wr, r) = padded(60, rows_a, cols_a), padded(61, rows_b, cols_b, 0.2), padded(62, M, N)
    wc = util.normal(63, batch * (N + 5)).reshape(batch, N + 5)
    wy = np.full_like(wr, 7.0)
    dA, dB, dR, dC, dY = (util.to_dev(t) for t in (wa, wb, wr, wc, wy))
    d = R.GemmF32Desc()
    d.M, d.N, d.K, d.transA, d.transB, d.alpha, d.beta, d.batch = M, N, K, transA, transB, 0.5, 1.0, batch
    d.A, d.B, d.C, d.Y, d.residual, d.bias_mode = util.ptr(dA), util.ptr(dB), util.ptr(dC), util.ptr(dY), util.ptr(dR), R.BIAS_ROW
    d.lda, d.ldb, d.ldy = cols_a + gap, cols_b + gap, N + gap
    d.strideA, d.strideB, d.strideC, d.strideY = wa[0].size, wb[0].size, N + 5, wy[0].size
    torch.cuda.synchronize()
    rt.call("sofie_hip_gemm_f32", C.byref(d))
    rt.sync()
    got = util.to_host(dY)
    for z in range(batch):
        u, v = (a[z].T if transA else a[z]).astype(np.float64), (b[z].T if transB else b[z]).astype(np.float64)
        want, most = 0.5 * (u @ v) + wc[z, :N] + r[z], 0.5 * (np.abs(u) @ np.abs(v)) + np.abs(wc[z, :N]) + np.abs(r[z])
        assert np.all(np.abs(got[z, :M, :N] - want) <= 1e-5 * most)
    got[:, :M, :N] = 7.0
    assert np.array_equal(got, wy)


@pytest.mark.parametrize("tile", [0] + TILES, indirect=True)
@pytest.mark.parametrize("case", [(2, 6, 15, 17, 10, 6, 6, (2, 3, 3, 2), (2, 1), (1, 1), 2), (3, 2, 12, 40, 66, 1, 33, (0, 16, 0, 0), (1, 3), (1, 1), 1),
                                  (1, 8, 20, 19, 130, 7, 5, (6, 0, 0, 4), (1, 2), (2, 1), 1)])
def test_convolutions_with_windows_past_31_positions(rt, tile, case):
    N, Cc, H, W, Cout, kh, kw, pads, strides, dils, group = case
    X = util.uniform01(64, N * Cc * H * W).reshape(N, Cc, H, W)
    Wt = util.normal(65, Cout * (Cc // group) * kh * kw, 0.3).reshape(Cout, Cc // group, kh, kw)
    b = util.normal(66, Cout)
    d = conv_desc(N, Cc, H, W, Cout, kh, kw, pads, strides, dils, group)
    dX, dW, db, dY = util.to_dev(X), util.to_dev(Wt), util.to_dev(b), util.dev_empty((N, Cout, d.OH, d.OW), np.float32)
    torch.cuda.synchronize()
    rt.call("sofie_hip_conv_f32", C.byref(d), util.ptr(dX), util.ptr(dW), util.ptr(db), R.ACT_RELU, C.c_float(0), util.ptr(dY), None, None)
    rt.sync()
    want = ob.conv_f32(X, Wt, b, pads=pads, strides=strides, dils=dils, group=group, act=1)
    assert np.abs(util.to_host(dY) - want).max() <= 1e-5 * max(1.0, float(np.abs(want).max()))


@pytest.mark.parametrize("tile", [0] + TILES, indirect=True)
def test_volumes_with_windows_past_31_positions(rt, tile):
    N, Cc, sp, Cout, k, pads, strides, dils, group = 2, 4, (7, 9, 8), 70, (3, 4, 3), (1, 2, 0, 1, 1, 2), (1, 2, 1), (2, 1, 1), 2
    X = util.uniform01(67, N * Cc * int(np.prod(sp))).reshape(N, Cc, *sp)
    Wt = util.normal(68, Cout * (Cc // group) * int(np.prod(k)), 0.3).reshape(Cout, Cc // group, *k)
    out = [(sp[a] + pads[a] + pads[a + 3] - (dils[a] * (k[a] - 1) + 1)) // strides[a] + 1 for a in range(3)]
    d = R.Conv3dDesc()
    (d.N, d.C, d.D, d.H, d.W, d.Cout, d.kd, d.kh, d.kw) = (N, Cc, *sp, Cout, *k)
    d.pad, d.stride, d.dil = (C.c_int32 * 6)(*pads), (C.c_int32 * 3)(*strides), (C.c_int32 * 3)(*dils)
    d.group, d.OD, d.OH, d.OW = group, *out
    dX, dW, dY = util.to_dev(X), util.to_dev(Wt), util.dev_empty((N, Cout, *out), np.float32)
    torch.cuda.synchronize()
    rt.call("sofie_hip_conv3d_f32", C.byref(d), util.ptr(dX), util.ptr(dW), None, R.ACT_NONE, C.c_float(0), util.ptr(dY), None, None)
    rt.sync()
    want = ob.conv3d_f32(X, Wt, None, pads=pads, strides=strides, dils=dils, group=group, act=0)
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
