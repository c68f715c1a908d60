"""The tile store of the fp32 products, which makes each choice once for four columns: every bias, a residual, one activation, several and none, with columns that end
inside, at and behind four, and rows of results that do and do not start on 16 bytes."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu

ACTS = {R.ACT_NONE: lambda v: v, R.ACT_RELU: lambda v: np.maximum(v, 0), R.ACT_LEAKYRELU: lambda v: np.where(v >= 0, v, 0.1 * v), R.ACT_SIGMOID: lambda v: 1 / (1 + np.exp(-v)),
        R.ACT_TANH: np.tanh, R.ACT_GELU: lambda v: 0.5 * v * (1 + np.vectorize(__import__("math").erf)(v / np.sqrt(2))), R.ACT_ABS: np.abs}


@pytest.mark.parametrize("tile", [32, 62, 64, 128])
@pytest.mark.parametrize("N", [3, 32, 33, 66, 131])
@pytest.mark.parametrize("mode", [R.BIAS_NONE, R.BIAS_ROW, R.BIAS_COL, R.BIAS_SCALAR, R.BIAS_FULL])
def test_store(rt, opt, tile, N, mode):
    M, K = 70, 40
    A, B, res = util.normal(90, M * K).reshape(M, K), util.normal(91, N * K, 0.2).reshape(N, K), util.normal(92, M * N).reshape(M, N)
    c = util.normal(93, {R.BIAS_NONE: 1, R.BIAS_ROW: N, R.BIAS_COL: M, R.BIAS_SCALAR: 1, R.BIAS_FULL: M * N}[mode])
    added = {R.BIAS_NONE: 0.0, R.BIAS_ROW: c[None, :], R.BIAS_COL: c[:, None], R.BIAS_SCALAR: c[0], R.BIAS_FULL: 0.5 * c.reshape(M if mode == R.BIAS_FULL else 1, -1)}[mode]
    p = A.astype(np.float64) @ B.T.astype(np.float64)
    most = np.abs(A).astype(np.float64) @ np.abs(B).T.astype(np.float64) * 1.25 + np.abs(added) + np.abs(res)
    dA, dB, dC, dR = (util.to_dev(t) for t in (A, B, c, res))
    opt("f32_tile", tile)
    for act, (residual, post) in [(a, e) for a in ACTS for e in ((False, None), (True, R.ACT_NEG))]:
        dY = util.dev_empty((M, N), np.float32)
        d = R.GemmF32Desc()
        d.M, d.N, d.K, d.transB, d.alpha, d.beta, d.bias_mode, d.act, d.act_alpha, d.batch = M, N, K, 1, 1.25, 0.5, mode, act, 0.1, 1
        d.A, d.B, d.C, d.Y = util.ptr(dA), util.ptr(dB), util.ptr(dC), util.ptr(dY)
        if residual:
            d.residual = util.ptr(dR)
        ops = R.PostOps()
        if post is not None:
            ops.count, ops.op[0] = 1, post
            d.post = C.pointer(ops)
        torch.cuda.synchronize()
        rt.call("sofie_hip_gemm_f32", C.byref(d))
        rt.sync()
        want = ACTS[act](1.25 * p + added + (res if residual else 0)) * (-1 if post is not None else 1)
        # K + 3 roundings of at most 2^-24 of the magnitudes; no activation is steeper than 1.13, and each is within 4 ulp
        assert np.all(np.abs(util.to_host(dY) - want) <= 1.13 * (K + 3) * 2.0 ** -24 * most + 2.0 ** -21 * (np.abs(want) + 2.0 ** -3)), (act, residual)
