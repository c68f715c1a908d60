"""int8 convolutions of small networks: few input channels read as windows whatever the image and output sizes, and NHWC layers
whose channels are a multiple of 8 or 16 but no power of two of 64 or more (gathered by the general GEMM loop), at the edges:
rows of 8, windows beside the row, missing last pixels, channels and outputs that fill no block, groups, strides, dilations."""
import numpy as np
import pytest

from oracle import binding as ob
from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_conv_i8 import run_conv

pytestmark = pytest.mark.gpu


def check(rt, case, out, relu, x_layout, y_layout):
    N, Cc, H, W, Cout, kh, kw, pads, strides, dils, group = case
    X = util.int8_sym(301, N * Cc * H * W).reshape(N, Cc, H, W)
    Wt = util.int8_sym(302, Cout * (Cc // group) * kh * kw).reshape(Cout, Cc // group, kh, kw)
    bias = util.int32_range(303, Cout, -500, 500)
    K = (Cc // group) * kh * kw
    scale = ((0.5 + util.uniform01(304, Cout)) / np.float32(127.0 * np.sqrt(K))).astype(np.float32)
    want = ob.conv_i8(X, Wt, bias, scale, pads=pads, strides=strides, dils=dils, group=group, relu=relu, out=out, omp=True)
    got = run_conv(rt, X, Wt, bias, scale, case, relu, out, x_layout, y_layout, 1)
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("case", [
    (3, 3, 9, 8, 16, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),
    (1, 1, 8, 9, 5, 3, 4, (0, 5, 0, 6), (1, 1), (1, 1), 1),      # windows wholly beside the row on both sides
    (2, 3, 21, 19, 24, 3, 3, (1, 1, 1, 1), (2, 2), (1, 1), 1),
    (2, 4, 10, 33, 33, 4, 2, (2, 0, 1, 1), (1, 3), (2, 1), 1),
    (5, 3, 28, 28, 64, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),
    (2, 6, 12, 17, 20, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 2),
    (90, 1, 30, 31, 32, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),  # more groups of pixels than waves
])
@pytest.mark.parametrize("out,relu", [(R.I8OUT_I8, 1), (R.I8OUT_F32, 0)])
@pytest.mark.parametrize("y_layout", [R.LAYOUT_NCHW, R.LAYOUT_NHWC])
def test_few_input_channels(rt, case, out, relu, y_layout):
    check(rt, case, out, relu, R.LAYOUT_NCHW, y_layout)


@pytest.mark.parametrize("case", [
    (2, 8, 9, 9, 24, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),
    (3, 16, 13, 11, 33, 3, 3, (1, 1, 1, 1), (2, 1), (1, 2), 1),
    (2, 24, 14, 14, 64, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),
    (1, 32, 17, 16, 130, 5, 5, (2, 2, 2, 2), (1, 1), (1, 1), 1),
    (2, 40, 8, 9, 16, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), 1),
    (2, 96, 10, 10, 48, 3, 3, (0, 1, 1, 0), (1, 1), (1, 1), 2),
])
@pytest.mark.parametrize("out,relu", [(R.I8OUT_I8, 1), (R.I8OUT_I32, 0)])
def test_channels_in_multiples_of_eight(rt, case, out, relu):
    check(rt, case, out, relu, R.LAYOUT_NHWC, R.LAYOUT_NHWC)


@pytest.mark.parametrize("N,Cc,HW", [(1, 16, 1), (3, 48, 63), (5, 64, 784), (2, 272, 100), (70, 16, 65)])
def test_global_average_of_int8_maps(rt, N, Cc, HW):
    import ctypes as C
    import torch
    X = util.int8_sym(305, N * HW * Cc).reshape(N, HW, Cc)
    dX, dY = util.to_dev(X), util.dev_empty((N, Cc), np.float32)
    torch.cuda.synchronize()
    rt.call("sofie_hip_global_avg_pool_i8", util.ptr(dY), util.ptr(dX), N, Cc, HW, R.LAYOUT_NHWC, C.c_float(0.05))
    rt.sync()
    want = (X.astype(np.int64).sum(axis=1).astype(np.float32) * np.float32(0.05)) / np.float32(HW)
    assert np.array_equal(util.to_host(dY), want)
