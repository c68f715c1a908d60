"""Values of the option "i8_tile" that name a kernel for other convolutions (27: few input channels; 17 and 33: small layers whose results are stored) or for products (164): a convolution that
the kernel does not take is left to the others, whichever way it reads its input.  Bit for bit."""
import numpy as np
import pytest

from oracle import binding as ob
from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_conv_i8 import run_conv, run_conv_plane_sums

pytestmark = pytest.mark.gpu


def layer(seed, case):
    N, Cc, H, W, Cout, kh, kw, pads, strides, dils, group = case
    X, Wt = util.int8_sym(seed, N * Cc * H * W).reshape(N, Cc, H, W), util.int8_sym(seed + 1, Cout * (Cc // group) * kh * kw).reshape(Cout, Cc // group, kh, kw)
    bias = util.int32_range(seed + 2, Cout, -2000, 2000)
    scale = ((0.5 + util.uniform01(seed + 3, Cout)) / np.float32(127.0 * np.sqrt(Wt[0].size))).astype(np.float32)
    return X, Wt, bias, scale


@pytest.mark.parametrize("tile", [17, 33, 27, 164])
@pytest.mark.parametrize("case, x_layout", [
    ((3, 64, 16, 16, 128, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1), R.LAYOUT_NHWC),     # input read directly
    ((2, 128, 32, 32, 96, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), 2), R.LAYOUT_NHWC),     # in groups
    ((4, 3, 16, 32, 40, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1), R.LAYOUT_NCHW),       # gathered
])
def test_plane_sums(rt, opt, tile, case, x_layout):
    pads, strides, dils, group = case[7:]
    X, Wt, bias, scale = layer(400 + tile, case)
    opt("i8_tile", tile)
    sums, _ = run_conv_plane_sums(rt, X, Wt, bias, scale, case, 1, x_layout)
    fmap = ob.conv_i8(X, Wt, bias, scale, pads=pads, strides=strides, dils=dils, group=group, relu=1, out=2, omp=True)
    assert np.array_equal(sums, fmap.astype(np.int64).sum(axis=(2, 3)))


@pytest.mark.parametrize("tile", [17, 33, 27, 164])
@pytest.mark.parametrize("case, x_layout", [
    ((2, 64, 12, 11, 64, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1), R.LAYOUT_NHWC),      # input read directly
    ((2, 48, 9, 10, 40, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1), R.LAYOUT_NHWC),       # gathered in the general loop
    ((2, 48, 9, 10, 40, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1), R.LAYOUT_NCHW),       # a column matrix
    ((3, 3, 14, 13, 24, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1), R.LAYOUT_NCHW),       # few channels
])
def test_results(rt, opt, tile, case, x_layout):
    pads, strides, dils, group = case[7:]
    X, Wt, bias, scale = layer(500 + tile, case)
    opt("i8_tile", tile)
    want = ob.conv_i8(X, Wt, bias, scale, pads=pads, strides=strides, dils=dils, group=group, relu=1, out=2, omp=True)
    assert np.array_equal(run_conv(rt, X, Wt, bias, scale, case, 1, R.I8OUT_I8, x_layout, R.LAYOUT_NHWC, 1), want)
