"""fp32 3 x 3 convolutions of up to four input channels: the tiles of 128 pixels that run through images (f32_conv3x3.hpp, four channels wide) and the choice between them and the kernel
whose workgroups stay within an image (f32_conv3x3_few.hpp)."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_conv3x3_split import products, run, tile  # noqa: F401 (a fixture)
from tests.test_gpu_f32 import conv_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [0, 3128], indirect=True)
@pytest.mark.parametrize("channels, out, images, H, W, pads, group", [
    (1, 1, 1, 3, 3, (0, 0, 0, 0), 1), (4, 64, 700, 3, 3, (1, 1, 1, 1), 1), (3, 33, 257, 4, 4, (1, 1, 1, 1), 1), (2, 31, 130, 5, 7, (1, 0, 2, 1), 1), (4, 32, 64, 4, 8, (1, 1, 1, 1), 1),
    (3, 70, 9, 11, 13, (2, 1, 1, 2), 1), (4, 17, 3, 33, 2, (1, 1, 1, 1), 1), (6, 10, 40, 6, 5, (1, 1, 1, 1), 2), (5, 5, 90, 3, 4, (1, 1, 1, 1), 5), (3, 65, 2, 5, 115, (1, 1, 1, 1), 1)])
def test_tiles_through_images(rt, tile, channels, out, images, H, W, pads, group):
    seed = 200 + 10 * (tile != 0)
    X, Wt = util.normal(seed, images * channels * H * W).reshape(images, channels, H, W), util.normal(seed + 1, out * channels // group * 9, 0.3).reshape(out, channels // group, 3, 3)
    p = products(X, Wt, pads, group)
    b, r = util.normal(seed + 2, out), util.normal(seed + 3, p[..., 0].size).reshape(p.shape[:4])
    for bias, residual, act in ((b, r, R.ACT_RELU), (None, None, R.ACT_NONE), (b, None, R.ACT_LEAKYRELU)):
        got = run(rt, X, Wt, bias, pads, group, act=act, residual=residual)
        want, most = p.sum(4), np.abs(p).sum(4)
        for extra in (bias.reshape(1, -1, 1, 1) if bias is not None else 0, residual if residual is not None else 0):
            want, most = want + extra, most + np.abs(extra)
        want = np.where(want >= 0, want, want * {R.ACT_RELU: 0.0, R.ACT_NONE: 1.0, R.ACT_LEAKYRELU: np.float64(np.float32(0.1))}[act])
        # an instruction per two products at least, each within 2 2^-24 of the magnitudes so far, then bias, residual and activation
        assert np.all(np.abs(got - want) <= (2 * 9 * channels // group // 2 + 8) * 2.0 ** -24 * most)


@pytest.mark.parametrize("images, channels, H, W, out", [(16384, 4, 3, 3, 64), (16384, 3, 5, 5, 32), (2048, 4, 8, 8, 64), (136, 4, 24, 10, 118), (64, 3, 64, 64, 32), (512, 1, 28, 28, 32)])
def test_the_faster_kernel_is_chosen(rt, opt, images, channels, H, W, out):
    """The choice costs at most 15 % where it was fitted; the slower kernel takes 1.2 to 9 times as long here."""
    d = conv_desc(images, channels, H, W, out, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1)
    dX, dW, dY = torch.randn(images * channels * H * W, device="cuda"), torch.randn(out * channels * 9, device="cuda"), torch.empty(images * out * H * W, device="cuda")
    torch.cuda.synchronize()

    def us(kernel):
        opt("f32_tile", kernel)
        best = 1e9
        for again in range(7):
            rt.timer_start()
            for _ in range(20):
                rt.call("sofie_hip_conv_f32", C.byref(d), util.ptr(dX), util.ptr(dW), None, R.ACT_NONE, C.c_float(0.0), util.ptr(dY), None, None)
            best = min(best, rt.timer_stop() * 1e3 / 20)
        return best
    us(0)   # the card awake
    chosen, within, through = us(0), us(3004), us(3128)
    print(chosen, within, through, flush=True)
    assert chosen <= 1.2 * min(within, through)
