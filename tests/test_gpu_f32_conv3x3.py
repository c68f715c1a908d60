"""The fp32 3 x 3 convolution with its patch in LDS, every tile forced by the context option "f32_tile": tiles that begin and end in the
middle of a row, that run through several images, patches of few and of many columns, paddings of none, one and two (and not
the same on both sides), channels that are no multiple of a slab, weights with and without 16-byte rows, output channels around a
tile, groups, a residual."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import binding as ob
from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_f32 import conv_desc
from tests.test_gpu_f32_tiles import conv2d_f64

pytestmark = pytest.mark.gpu

CASES = [
    # images, channels, H, W, channels out, pads, group
    (2, 8, 16, 32, 64, (1, 1, 1, 1), 1),      # rows divide the tile
    (7, 16, 6, 5, 33, (1, 1, 1, 1), 1),       # several images per tile
    (3, 20, 13, 11, 65, (1, 1, 1, 1), 1),     # half a slab, one column past a tile
    (2, 9, 17, 23, 18, (0, 0, 0, 0), 1),      # weights of 81 floats a row
    (1, 13, 20, 96, 40, (1, 2, 2, 0), 1),     # wide rows, paddings of their own
    (3, 10, 27, 60, 34, (1, 1, 1, 1), 1),     # patches of two rows and of four
    (2, 8, 95, 95, 16, (1, 1, 1, 1), 1),      # the widest, through the edge of an image
    (2, 3, 31, 30, 37, (1, 1, 1, 1), 1),      # a colour image
    (3, 1, 12, 12, 8, (1, 1, 1, 1), 1),
    (2, 24, 9, 14, 20, (1, 1, 1, 1), 2),      # groups of 12 -> 10
    (130, 5, 3, 3, 4, (0, 0, 0, 0), 1),       # one pixel per image
]


@pytest.mark.parametrize("tile", [0, 3032, 3064, 3128])
@pytest.mark.parametrize("case", CASES)
def test_conv3x3(rt, tile, case):
    N, Cc, H, W, Cout, pads, group = case
    X = util.uniform01(40, N * Cc * H * W).reshape(N, Cc, H, W)
    Wt = util.normal(41, Cout * (Cc // group) * 9, 0.3).reshape(Cout, Cc // group, 3, 3)
    b = util.normal(42, Cout)
    d = conv_desc(N, Cc, H, W, Cout, 3, 3, pads, (1, 1), (1, 1), group)
    res = util.normal(43, N * Cout * d.OH * d.OW).reshape(N, Cout, d.OH, d.OW)
    dX, dW, db, dR, dY = util.to_dev(X), util.to_dev(Wt), util.to_dev(b), util.to_dev(res), util.dev_empty(res.shape, np.float32)
    torch.cuda.synchronize()
    print("conv3x3", tile, case, flush=True)
    rt.set_option("f32_tile", tile)
    try:
        for residual in (None, util.ptr(dR)):
            rt.call("sofie_hip_conv_f32", C.byref(d), util.ptr(dX), util.ptr(dW), util.ptr(db), R.ACT_RELU, C.c_float(0), util.ptr(dY), None, residual)
            rt.sync()
            want = ob.conv_f32(X, Wt, b, pads=pads, strides=(1, 1), dils=(1, 1), group=group, act=0)
            want = np.maximum(want + (res if residual else 0), 0)
            assert np.abs(util.to_host(dY) - want).max() <= 1e-5 * max(1.0, float(np.abs(want).max()))
    finally:
        rt.set_option("f32_tile", 0)


@pytest.mark.parametrize("tile", [0, 3032, 3064, 3128, 16, 62, 64, 126])
@pytest.mark.parametrize("channels", [3, 16, 200])
@pytest.mark.parametrize("bias, residual", [(1000.0, 0.0), (0.1, 1000.0), (700.0, 700.0)])
def test_bias_and_residual_are_rounded_once(rt, opt, tile, channels, bias, residual):
    """Beside a large bias or residual the products' sum keeps its own precision: the result is that sum plus two additions, each rounded once."""
    N, H, W, Cout = 2, 12, 17, 34
    X = util.uniform01(44, N * channels * H * W).reshape(N, channels, H, W)
    Wt = util.normal(45, Cout * channels * 9, 0.1).reshape(Cout, channels, 3, 3)
    b, r = util.normal(46, Cout, bias), util.normal(47, N * Cout * H * W, residual or 1.0).reshape(N, Cout, H, W) * np.float32(residual != 0)
    d = conv_desc(N, channels, H, W, Cout, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1)
    dX, dW, db, dR, dY = util.to_dev(X), util.to_dev(Wt), util.to_dev(b), util.to_dev(r), util.dev_empty(r.shape, np.float32)
    torch.cuda.synchronize()
    opt("f32_tile", tile)
    rt.call("sofie_hip_conv_f32", C.byref(d), util.ptr(dX), util.ptr(dW), util.ptr(db), R.ACT_NONE, C.c_float(0), util.ptr(dY), None, util.ptr(dR))
    rt.sync()
    products, most = conv2d_f64(X, Wt, (1, 1, 1, 1))
    beside = np.abs(b.astype(np.float64))[None, :, None, None] + np.abs(r)
    # two additions of values below `beside` + most; 1800 products summed in any order stay far within 1e-6 of their magnitudes
    assert np.all(np.abs(util.to_host(dY) - (products + b[None, :, None, None] + r)) <= 2 * 2.0 ** -24 * (beside + most) + 1e-6 * most)
