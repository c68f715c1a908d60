"""Pooling of 3 x 3 windows with strides of two, a pair of results per thread and the left column from the lane before: rows of two and three columns, odd and even
extents, rows that end and begin inside a wave, every padding that takes this route and the first that does not, NaN and infinities.  The bits of the
reference's loops."""
import numpy as np
import pytest

from tests import util
from tests.test_gpu_pool import both, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["max", "average"])
@pytest.mark.parametrize("H, W", [(3, 3), (2, 2), (1, 3), (5, 4), (4, 63), (7, 128), (3, 129), (31, 130)])
@pytest.mark.parametrize("pads", [[1, 1, 1, 1], [0, 0, 2, 2], [2, 1, 1, 2], [1, 2, 1, 0]])
def test_pool_step2(rt, mode, H, W, pads):
    X = util.normal(9110, 7 * H * W).reshape(1, 7, H, W)
    X.reshape(-1)[[0, H * W // 2, -1]] = np.nan, np.inf, -np.inf
    for ceil in (0, 1):
        if H + pads[0] + pads[2] < 3 or W + pads[1] + pads[3] < 3:
            continue
        with np.errstate(invalid="ignore"):
            got, want = both(rt, X, mode, [3, 3], pads, [2, 2], None, "NOTSET", ceil, ceil)
        assert got.shape == want.shape and np.array_equal(np.isnan(got), np.isnan(want))
        assert same_bits(np.where(np.isnan(got), np.float32(0), got), np.where(np.isnan(want), np.float32(0), want))
