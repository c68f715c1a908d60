"""The int8 / FP8 kernel for few rows whose operands pass through a ring in LDS (rows on 16 bytes), at the edges of its tiles (16 and 32), of its steps of
128 bytes of k over eight waves, and of its ring (four or two places; fewer where there are more tiles than CUs): less than a step, a chunk more or less than
whole steps, more steps than the rings hold, rows that lie further apart than they are long."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import binding as ob
from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 16, 0), (16, 17, 112, 16), (31, 33, 128, 0), (17, 15, 144, 48), (33, 64, 1040, 0), (5, 40, 4096, 16), (48, 20, 4240, 0), (16, 16, 9200, 0), (300, 600, 400, 0), (270, 530, 2064, 16),
          # by registers: whole steps up to 256 bytes (of 32 x 32 tiles two a CU, and more than that by lines), four rows up to 768
          (33, 70, 256, 16), (16, 16, 128, 0), (500, 1040, 128, 0), (530, 1040, 256, 16), (4, 48, 768, 0), (5, 48, 768, 16), (3, 33, 896, 0), (2, 20, 384, 0)]


@pytest.fixture
def tile(rt, request):
    for name in ("i8_tile", "f8_tile"):
        rt.set_option(name, request.param)
    yield request.param
    for name in ("i8_tile", "f8_tile"):
        rt.set_option(name, 0)


def padded(rows, gap, filler):
    whole = np.full((rows.shape[0], rows.shape[1] + gap), filler, rows.dtype)
    whole[:, :rows.shape[1]] = rows
    return util.to_dev(whole)


@pytest.mark.parametrize("tile", [0, 16, 32], indirect=True)
@pytest.mark.parametrize("M,N,K,gap", SHAPES)
def test_int8(rt, tile, M, N, K, gap):
    A, B = util.int8_sym(80, M * K).reshape(M, K), util.int8_sym(81, N * K).reshape(N, K)
    dA, dB, dY = padded(A, gap, 127), padded(B, gap, -127), util.dev_empty((M, N), np.int32)
    d = R.GemmI8Desc()
    d.M, d.N, d.K, d.transB, d.out, d.lda, d.ldb = M, N, K, 1, R.I8OUT_I32, K + gap, K + gap
    d.A, d.B, d.Y = util.ptr(dA), util.ptr(dB), util.ptr(dY)
    d.scale_scalar = d.q_scale = 1.0
    torch.cuda.synchronize()
    rt.call("sofie_hip_gemm_i8", C.byref(d))
    rt.sync()
    assert np.array_equal(util.to_host(dY), A.astype(np.int64) @ B.astype(np.int64).T)


@pytest.mark.parametrize("tile", [0, 16, 32], indirect=True)
@pytest.mark.parametrize("M,N,K,gap", SHAPES)
def test_fp8(rt, tile, M, N, K, gap):
    A, B = (ob.quantize_fp8(util.normal(s, r * K).reshape(r, K), 1.0) for s, r in ((82, M), (83, N)))
    dA, dB, dY = padded(A, gap, 0x7f), padded(B, gap, 0x7f), util.dev_empty((M, N), np.float32)    # 0x7f: NaN
    d = R.GemmFp8Desc()
    d.M, d.N, d.K, d.transB, d.scale, d.out, d.lda, d.ldb = M, N, K, 1, 0.5, R.F8OUT_F32, K + gap, K + gap
    d.A, d.B, d.Y = util.ptr(dA), util.ptr(dB), util.ptr(dY)
    torch.cuda.synchronize()
    rt.call("sofie_hip_gemm_fp8", C.byref(d))
    rt.sync()
    a, b = ob.e4m3_to_f32(A).astype(np.float64), ob.e4m3_to_f32(B).astype(np.float64).T
    # the bound of the other FP8 products: fp32 sums in the matrix cores' own order
    assert np.all(np.abs(util.to_host(dY) - 0.5 * (a @ b)) <= 2.0 ** -14 * 0.5 * (np.abs(a) @ np.abs(b)) + 1e-12)
