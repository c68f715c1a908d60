"""The fp32 kernel for small products whose operands pass through a ring in LDS (both contiguous in k, rows on 16 bytes), at the edges of its tile (16), of its
steps of 32 k over eight waves and of its ring: up to a step (by registers), four k more or less than whole steps, more steps than the ring holds, more tiles than CUs,
batches, and rows that lie further apart than they are long."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,gap,batch", [(1, 1, 4, 0, 1), (16, 17, 28, 4, 1), (31, 15, 32, 0, 2), (17, 16, 36, 12, 3), (5, 33, 260, 0, 1), (16, 16, 1024, 4, 1), (33, 20, 1060, 0, 2),
                                             (16, 31, 2300, 0, 1), (300, 300, 132, 0, 1), (40, 70, 516, 8, 30)])
def test_products(rt, M, N, K, gap, batch):
    def padded(seed, rows, scale):
        whole = np.full((batch, rows, K + gap), np.nan, np.float32)
        whole[:, :, :K] = util.normal(seed, batch * rows * K, scale).reshape(batch, rows, K)
        return util.to_dev(whole), whole[:, :, :K].astype(np.float64)
    (dA, a), (dB, b) = padded(90, M, 1.0), padded(91, N, 0.2)
    bias = util.normal(92, N)
    db, dY = util.to_dev(bias), util.dev_empty((batch, M, N), np.float32)
    d = R.GemmF32Desc()
    d.M, d.N, d.K, d.transB, d.alpha, d.beta, d.batch, d.lda, d.ldb = M, N, K, 1, 1.5, 1.0, batch, K + gap, K + gap
    d.A, d.B, d.C, d.Y, d.bias_mode = util.ptr(dA), util.ptr(dB), util.ptr(db), util.ptr(dY), R.BIAS_ROW
    d.strideA, d.strideB, d.strideY = M * (K + gap), N * (K + gap), M * N
    rt.set_option("f32_tile", 16)
    try:
        torch.cuda.synchronize()
        rt.call("sofie_hip_gemm_f32", C.byref(d))
        rt.sync()
    finally:
        rt.set_option("f32_tile", 0)
    want = 1.5 * (a @ b.transpose(0, 2, 1)) + bias
    # products and additions rounded once each: one chain of four k per MFMA and 16 per step over a wave's steps, then sixteen parts, alpha and the bias
    n = 4 * -(-K // 256) * 4 + 16 + 4
    assert np.all(np.abs(util.to_host(dY) - want) <= n * 2.0 ** -24 * (1.5 * (np.abs(a) @ np.abs(b).transpose(0, 2, 1)) + np.abs(bias)))
