"""The direct kernel of small int8 convolutions over NHWC input (conv_i8_direct.hpp), forced by the option "i8_tile" and as chosen: tiles of 16 and 32 pixels and channels that are not
filled, reductions of one piece, of a step of 128 bytes and around it, of more steps than the four waves have at once, pieces of 8 and 16 bytes, strides, dilations, paddings of
their own, groups, both layouts of the result.  Bit for bit."""
import pytest

from sofie_amd import runtime as R
from tests.test_gpu_conv_i8_small_layers import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [0, 17, 33])
@pytest.mark.parametrize("case", [
    (1, 8, 1, 1, 1, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), 1),
    (3, 8, 5, 7, 15, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),        # 72 bytes of k
    (2, 128, 4, 5, 17, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), 1),      # one whole step
    (2, 144, 5, 5, 31, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), 1),
    (5, 16, 11, 9, 33, 3, 3, (1, 0, 2, 1), (2, 1), (1, 2), 1),
    (1, 24, 13, 6, 64, 5, 4, (2, 1, 2, 3), (1, 3), (2, 1), 1),
    (2, 64, 9, 8, 48, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),
    (1, 256, 6, 7, 20, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),      # 18 steps
    (2, 48, 6, 6, 42, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 3),
    (2, 128, 6, 6, 36, 3, 3, (1, 1, 1, 1), (2, 2), (1, 1), 2),
])
@pytest.mark.parametrize("out,relu,y_layout", [(R.I8OUT_I8, 1, R.LAYOUT_NHWC), (R.I8OUT_F32, 0, R.LAYOUT_NCHW), (R.I8OUT_I32, 1, R.LAYOUT_NHWC)])
def test_small_layers(rt, opt, tile, case, out, relu, y_layout):
    opt("i8_tile", tile)
    check(rt, case, out, relu, R.LAYOUT_NHWC, y_layout)
