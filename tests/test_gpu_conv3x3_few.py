"""The fp32 3 x 3 convolution of up to four input channels (f32_conv3x3_few.hpp): reductions of 9 to 36 products padded to a multiple of four, output channels around its blocks
of 16 and its tiles of four of them, images of fewer pixels than a workgroup takes and of any number more, paddings of their own, groups, with and without what is added."""
import numpy as np
import pytest

from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_conv3x3_split import products, run, tile  # noqa: F401 (a fixture)
from tests.test_gpu_f32_tiles import same_as_ieee, with_nonfinite

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [0, 3004], indirect=True)
@pytest.mark.parametrize("channels, out, images, H, W, pads, group", [
    (1, 1, 1, 3, 3, (0, 0, 0, 0), 1), (1, 17, 3, 12, 12, (1, 1, 1, 1), 1), (2, 16, 5, 9, 15, (1, 0, 2, 1), 1), (3, 8, 2, 31, 33, (1, 1, 1, 1), 1),
    (3, 33, 1, 7, 96, (1, 1, 1, 1), 1), (3, 48, 2, 16, 64, (2, 2, 2, 2), 1), (4, 63, 3, 13, 10, (1, 1, 1, 1), 1), (4, 64, 1, 6, 21, (0, 1, 1, 0), 1),
    (3, 65, 2, 11, 13, (1, 1, 1, 1), 1), (2, 130, 1, 8, 8, (1, 1, 1, 1), 1), (6, 10, 2, 17, 19, (1, 1, 1, 1), 2), (5, 5, 3, 14, 9, (1, 1, 1, 1), 5),
    (3, 4, 150, 5, 5, (1, 1, 1, 1), 1), (1, 2, 520, 20, 53, (1, 1, 1, 1), 1), (3, 2, 1, 4, 630, (1, 1, 1, 1), 1), (1, 1, 1, 5, 2558, (1, 1, 1, 1), 1)])
def test_few_channels(rt, tile, channels, out, images, H, W, pads, group):
    X, Wt = util.normal(90, images * channels * H * W).reshape(images, channels, H, W), util.normal(91, out * channels // group * 9, 0.3).reshape(out, channels // group, 3, 3)
    p = products(X, Wt, pads, group)
    b, r = util.normal(92, out), util.normal(93, p[..., 0].size).reshape(p.shape[:4])
    for bias, residual, act in ((b, r, R.ACT_RELU), (None, None, R.ACT_NONE), (b, None, R.ACT_LEAKYRELU)):
        got = run(rt, X, Wt, bias, pads, group, act=act, residual=residual)
        want, most = p.sum(4), np.abs(p).sum(4)
        for extra in (bias.reshape(1, -1, 1, 1) if bias is not None else 0, residual if residual is not None else 0):
            want, most = want + extra, most + np.abs(extra)
        want = np.where(want >= 0, want, want * {R.ACT_RELU: 0.0, R.ACT_NONE: 1.0, R.ACT_LEAKYRELU: np.float64(np.float32(0.1))}[act])
        # an instruction per four products, each within 2 2^-24 of the magnitudes so far, then bias, residual and activation
        assert np.all(np.abs(got - want) <= (2 * 9 * channels // group // 4 + 8) * 2.0 ** -24 * most)


@pytest.mark.parametrize("tile", [3004], indirect=True)
@pytest.mark.parametrize("channels", [1, 2, 3])
def test_nan_and_infinity(rt, tile, channels):
    """What pads the reduction is zero on both sides."""
    X, Wt = with_nonfinite(util.normal(94, 2 * channels * 13 * 11), 95).reshape(2, channels, 13, 11), util.normal(96, 5 * channels * 9).reshape(5, channels, 3, 3)
    with np.errstate(invalid="ignore"):
        p = products(X, Wt, (1, 1, 1, 1))
        same_as_ieee(run(rt, X, Wt, None, (1, 1, 1, 1)), p.sum(4), np.abs(p).sum(4))
