"""How the fp32 3 x 3 convolutions load what is added to a block's sums and store the block: output channels around the four that a lane holds side by side and
the 32 of a tile, with and without bias and residual, with one activation, none and a chain, and results that no buffer of 2 GiB holds."""
import numpy as np
import pytest
import torch
import ctypes as C

from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_conv3x3_split import products, roundings, run, tile  # noqa: F401 (a fixture)
from tests.test_gpu_f32 import conv_desc

pytestmark = pytest.mark.gpu
TILES = [3032, 3064, 3128, 4128, 4256]


@pytest.mark.parametrize("tile", TILES, indirect=True)
@pytest.mark.parametrize("channels", [3, 17])
@pytest.mark.parametrize("out", [1, 4, 5, 8, 11, 31, 32, 36, 59])
def test_output_channels(rt, tile, channels, out):
    H, W = (17, 16) if tile == 4256 else (9, 7)   # images that the kernel takes
    X, Wt = util.normal(80, 3 * channels * H * W).reshape(3, channels, H, W), util.normal(81, out * channels * 9, 0.3).reshape(out, channels, 3, 3)
    p = products(X, Wt, (1, 1, 1, 1))
    b, r = util.normal(82, out), util.normal(83, p[..., 0].size).reshape(p.shape[:4])
    for bias, residual, act in ((b, r, R.ACT_RELU), (None, r, R.ACT_NONE), (b, None, R.ACT_LEAKYRELU)):
        got = run(rt, X, Wt, bias, (1, 1, 1, 1), act=act, residual=residual)
        want, most = p.sum(4), np.abs(p).sum(4)
        for extra in (bias.reshape(1, -1, 1, 1) if bias is not None else 0, residual if residual is not None else 0):
            want, most = want + extra, most + np.abs(extra)
        want = np.where(want >= 0, want, want * {R.ACT_RELU: 0.0, R.ACT_NONE: 1.0, R.ACT_LEAKYRELU: np.float64(np.float32(0.1))}[act])
        # and bias, residual and activation
        n = roundings(tile, channels, H, W) if tile > 4000 else 2 * (9 * channels // 2 + 4)
        assert np.all(np.abs(got - want) <= (n + 3) * 2.0 ** -24 * most)


@pytest.mark.parametrize("tile", [3128, 4128], indirect=True)
def test_results_beyond_a_buffer(rt, tile):
    """1.1 GB of results per image: addresses of 64 bits."""
    channels, H, W, out = 3, 8192, 64, 523
    X, Wt, b = util.normal(84, channels * H * W).reshape(1, channels, H, W), util.normal(85, out * channels * 9, 0.3).reshape(out, channels, 3, 3), util.normal(86, out)
    d = conv_desc(1, channels, H, W, out, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1)
    dX, dW, db = util.to_dev(X), util.to_dev(Wt), util.to_dev(b)
    dR = torch.arange(out * H * W, dtype=torch.int32, device="cuda").remainder_(1021).float()
    dY = torch.full((out, H, W), float("nan"), device="cuda")
    torch.cuda.synchronize()
    rt.call("sofie_hip_conv_f32", C.byref(d), util.ptr(dX), util.ptr(dW), util.ptr(db), R.ACT_NONE, C.c_float(0), util.ptr(dY), None, util.ptr(dR))
    rt.sync()
    assert not bool(torch.isnan(dY).any())
    for rows in (slice(0, 6), slice(H - 6, H)):
        x = np.zeros((1, channels, 8, W), np.float32)
        x[0, :, 1:7] = X[0, :, rows]
        inner = slice(0, 5) if rows.start == 0 else slice(1, 6)   # the other row's neighbours are not among these
        p = products(x, Wt, (0, 1, 0, 1))[0]
        want = p.sum(3) + b[:, None, None] + dR.view(out, H, W)[:, rows].double().cpu().numpy()
        got = dY[:, rows].double().cpu().numpy()
        most = np.abs(p).sum(3) + np.abs(b)[:, None, None] + 1021
        assert np.all(np.abs(got - want)[:, inner] <= 2 * (9 * channels // 2 + 4 + 3) * 2.0 ** -24 * most[:, inner])
