"""The fp32 3 x 3 convolution that multiplies bf16 pieces (f32_conv3x3_split.hpp), forced by the context option "f32_tile", at the edges of its tiles (128 or 256
pixels, 32 output channels), of its slabs (16 channels) and of its patch (360 places), against sums in 64 bits: the error is that of fp32 sums, at any
scale of the inputs down to the smallest subnormal number, and infinities and NaN are where IEEE arithmetic has them."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util
from tests.test_gpu_f32 import conv_desc
from tests.test_gpu_f32_tiles import same_as_ieee, with_nonfinite

pytestmark = pytest.mark.gpu


@pytest.fixture
def tile(rt, request):
    rt.set_option("f32_tile", request.param)
    yield request.param
    rt.set_option("f32_tile", 0)


def run(rt, X, Wt, b, pads, group=1, act=R.ACT_NONE, residual=None):
    N, Cc, H, W = X.shape
    d = conv_desc(N, Cc, H, W, len(Wt), 3, 3, pads, (1, 1), (1, 1), group)
    dX, dW, dY = util.to_dev(X), util.to_dev(Wt), util.dev_empty((N, len(Wt), d.OH, d.OW), np.float32)
    db, dR = (util.to_dev(t) if t is not None else None for t in (b, residual))
    torch.cuda.synchronize()
    ptr = lambda t: util.ptr(t) if t is not None else None
    rt.call("sofie_hip_conv_f32", C.byref(d), ptr(dX), ptr(dW), ptr(db), act, C.c_float(0.1), ptr(dY), None, ptr(dR))
    rt.sync()
    return util.to_host(dY)


def products(X, Wt, pads, group=1):
    """Every product of every sum, in 64 bits: [image, output channel, row, column, k]."""
    x = np.pad(X.astype(np.float64), ((0, 0), (0, 0), (pads[0], pads[2]), (pads[1], pads[3])))
    win = np.lib.stride_tricks.sliding_window_view(x, (3, 3), axis=(2, 3)).transpose(0, 2, 3, 1, 4, 5)
    Cg, Ng = Wt.shape[1], len(Wt) // group
    parts = [win[:, None, :, :, g * Cg:(g + 1) * Cg] * Wt[g * Ng:(g + 1) * Ng].astype(np.float64)[None, :, None, None] for g in range(group)]
    whole = np.concatenate(parts, axis=1)
    return whole.reshape(*whole.shape[:4], -1)


def in_pieces(tile, OH, OW):
    """Whether the kernel takes images of OH x OW results at this tile: its patch, the rows a tile touches, two more and two per image that it runs into, is at most
    360 places.  256 pixels: of 8, 16 or 32 columns."""
    bm, plane = tile - 4000, OH * OW
    rows = bm // OW if bm % OW == 0 else (bm - 2 + OW) // OW + 1
    images = 0 if plane % bm == 0 else (bm - 2 + plane) // plane
    return (rows + 2 + 2 * images) * (OW + 2) <= 360


def roundings(tile, Cg, OH, OW):
    """Errors of a sum, in 2^-24 of the sum of magnitudes.  In pieces: an instruction per 16 channels and kernel position for the leading products, each within 2 (1.6
    measured) of the magnitudes so far, seven for terms of at most 2^-7 of them together (2 2^-8 + 3 2^-16 + ...), and the join.  In fp32: one per two products."""
    return 2 * 9 * -(-Cg // 16) * (1 + 7 * 2.0 ** -7 * 1.02) + 1 if in_pieces(tile, OH, OW) else 2 * (9 * Cg // 2 + 4)


CASES = [(1, 1, 3, 3, 1, (1, 1, 1, 1), 1), (3, 15, 9, 7, 31, (0, 0, 0, 0), 1), (2, 17, 13, 11, 33, (1, 0, 2, 1), 1), (1, 32, 16, 16, 64, (1, 1, 1, 1), 1), (5, 36, 8, 33, 20, (1, 1, 1, 1), 1),
         (2, 20, 10, 12, 66, (2, 2, 2, 2), 2), (17, 16, 4, 4, 32, (1, 1, 1, 1), 1), (1, 33, 5, 118, 3, (1, 1, 1, 1), 1),
         # taken at 256 pixels: tiles across images, a last one that is not filled, odd channels, groups
         (3, 15, 17, 16, 31, (1, 1, 1, 1), 1), (1, 33, 18, 18, 20, (0, 0, 0, 0), 1), (2, 17, 24, 32, 33, (1, 1, 1, 1), 1), (2, 20, 34, 9, 66, (1, 0, 1, 1), 2)]


@pytest.mark.parametrize("tile", [4128, 4256], indirect=True)
@pytest.mark.parametrize("scale", [1.0, 1e-30, 1e30])
@pytest.mark.parametrize("case", CASES)
def test_convolutions_around_tile_edges(rt, tile, case, scale):
    N, Cc, H, W, Cout, pads, group = case
    X = (util.normal(70, N * Cc * H * W).reshape(N, Cc, H, W) * np.float32(scale)).astype(np.float32)
    Wt = util.normal(71, Cout * Cc // group * 9, 0.3).reshape(Cout, Cc // group, 3, 3)
    b = (util.normal(72, Cout) * np.float32(scale)).astype(np.float32)
    p = products(X, Wt, pads, group)
    r = (util.normal(73, p[..., 0].size) * np.float32(scale)).reshape(p.shape[:4]).astype(np.float32)
    got = run(rt, X, Wt, b, pads, group, R.ACT_LEAKYRELU, r)
    want = p.sum(4) + b.reshape(1, -1, 1, 1) + r
    most = np.abs(p).sum(4) + np.abs(b).reshape(1, -1, 1, 1) + np.abs(r)
    want = np.where(want >= 0, want, np.float64(np.float32(0.1)) * want)
    # bias, residual and activation: another rounding each
    assert np.all(np.abs(got - want) <= (roundings(tile, Cc // group, *p.shape[2:4]) + 3) * 2.0 ** -24 * most)


@pytest.mark.parametrize("tile", [4128, 4256], indirect=True)
@pytest.mark.parametrize("case", [(2, 18, 13, 11, 35), (1, 3, 40, 41, 5), (2, 19, 17, 16, 35)])
def test_nan_infinity_and_the_largest_numbers(rt, tile, case):
    N, Cc, H, W, Cout = case
    X = with_nonfinite(util.normal(74, N * Cc * H * W), 75).reshape(N, Cc, H, W)
    X.reshape(-1)[7] = np.finfo(np.float32).max            # rounds to an infinity in bf16
    Wt = util.normal(76, Cout * Cc * 9, 0.2).reshape(Cout, Cc, 3, 3)
    Wt[1, 0, 0, 0] = np.inf
    Wt[2] = np.clip(Wt[2], -0.9, 0.9)
    with np.errstate(invalid="ignore", over="ignore"):
        p = products(X, Wt, (1, 1, 1, 1))
        want, most = p.sum(4), np.abs(p).sum(4)
    got = run(rt, X, Wt, None, (1, 1, 1, 1))
    assert np.all(np.abs(want[np.isfinite(want)]) < np.finfo(np.float32).max)
    same_as_ieee(got, want, most)


SMALL = [(1e-33, 1e9), (1e-36, 1e12), (1e37, 1e-37), (3e-42, 1e30)]    # of the inputs, of the weights: results are normal numbers


@pytest.mark.parametrize("tile", [4128, 4256], indirect=True)
@pytest.mark.parametrize("scales", SMALL)
@pytest.mark.parametrize("case", [(3, 15, 9, 7, 31, (0, 0, 0, 0), 1), (2, 17, 13, 11, 33, (1, 0, 2, 1), 1), (2, 20, 10, 12, 66, (2, 2, 2, 2), 2), (17, 16, 4, 4, 32, (1, 1, 1, 1), 1),
                                  (3, 15, 17, 16, 31, (1, 1, 1, 1), 1), (2, 20, 34, 9, 66, (1, 0, 1, 1), 2)])
def test_numbers_that_pieces_do_not_hold(rt, tile, case, scales):
    """bf16 holds multiples of 2^-133: the last bits of values below 2^-110 (7.7e-34) are in no piece."""
    N, Cc, H, W, Cout, pads, group = case
    X = (util.normal(77, N * Cc * H * W).astype(np.float64) * scales[0]).astype(np.float32).reshape(N, Cc, H, W)
    Wt = (util.normal(78, Cout * Cc // group * 9, 0.3).astype(np.float64) * scales[1]).astype(np.float32).reshape(Cout, Cc // group, 3, 3)
    p = products(X, Wt, pads, group)
    got = run(rt, X, Wt, None, pads, group)
    # fp32 multiply-adds, two products at a time, each within 2^-23 of the magnitudes so far
    n = 9 * (Cc // group)
    assert np.all(np.abs(got - p.sum(4)) <= n * 2.0 ** -23 * np.abs(p).sum(4))
    # rounding errors cancel in part: a sequential fp32 sum comes to 0.45 of this, pieces cut at 2^-133 to 50 and more from 1e-36 on
    assert np.linalg.norm(got - p.sum(4)) <= 2.0 ** -21 * np.linalg.norm(p.sum(4))


def piece_rich(seed, n):
    """Numbers from 1 on whose second and third bf16 pieces are near their largest, 2^-8 and 2^-17 (and of either sign)."""
    sign = np.where(util.normal(seed, n) < 0, -1.0, 1.0)
    rest = 1 - np.abs(util.normal(seed + 1, n)) % 0.1, 1 - np.abs(util.normal(seed + 2, n)) % 0.1
    whole = 1 + np.floor(np.abs(util.normal(seed + 3, n)) % 1 * 8) / 128
    return (whole + 2.0 ** -8 * rest[0] * sign + 2.0 ** -17 * rest[1]).astype(np.float32)


@pytest.mark.parametrize("tile", [4128, 4256], indirect=True)
@pytest.mark.parametrize("channels", [16, 36])
def test_single_products(rt, tile, channels):
    """One nonzero weight per output channel, at every kernel position and in every slab: each result is one product, within 2^-24 of itself but for what the
    matrix cores lose of the small terms (seven sums of at most 2^-7 of it, 2^-23 of each) and the one left out (2^-34).  On the CPU, leaving out any one of the
    eight terms misses this by a quarter and more."""
    out = 9 * -(-channels // 4)
    X = piece_rich(90, 2 * channels * 342).reshape(2, channels, 19, 18)
    Wt, n = np.zeros((out, channels, 3, 3), np.float32), np.arange(out)
    Wt[n, (n // 9 * 4 + n % 4) % channels, n % 9 // 3, n % 3] = piece_rich(94, out)
    want = products(X, Wt, (0, 0, 0, 0)).sum(4)
    got = run(rt, X, Wt, None, (0, 0, 0, 0))
    assert np.all(np.abs(got - want) <= 2.0 ** -24 * (1 + 7 * 2.0 ** -6 + 2.0 ** -10) * np.abs(want))


@pytest.mark.parametrize("tile", [4128, 4256], indirect=True)
def test_one_small_number_that_counts(rt, tile):
    """Among ordinary numbers, one input and one weight that pieces cut, each the only thing in its sums."""
    X, Wt = util.normal(79, 2 * 18 * 272).reshape(2, 18, 17, 16), np.zeros((34, 18, 3, 3), np.float32)
    X[0, 17, 4, 4], X[:, 3] = np.float32(1.2345678e-37), 0
    Wt[33, 17, 1, 1] = np.float32(7.654321e35)             # 9.4e-2 at the one pixel, large numbers elsewhere
    Wt[5, 2, 0, 2] = np.float32(1.2345678e-38)
    X[1, 2] *= np.float32(1e37)
    p = products(X, Wt, (1, 1, 1, 1))
    got = run(rt, X, Wt, None, (1, 1, 1, 1))
    assert np.all(np.abs(got - p.sum(4)) <= 2.0 ** -23 * np.abs(p).sum(4) + 2.0 ** -149)
