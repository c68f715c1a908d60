"""The chain kernel's layers with W stored [N,K] in rows of 16 bytes: groups of 16, 32 and 64 lanes an output, at the edges of the groups (K = 64, 128) and of the pieces that a lane asks
for at once (256, 512), outputs around those of a pass (64, 128, 256), one, two and four rows a workgroup, the last one not filled, every kind of bias and a residual."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 66, 131])
@pytest.mark.parametrize("mode", [R.BIAS_NONE, R.BIAS_ROW, R.BIAS_COL, R.BIAS_SCALAR, R.BIAS_FULL])
@pytest.mark.parametrize("dims", [(4, 1, 64), (64, 257, 3), (68, 128, 65, 9), (132, 129, 4, 63), (512, 260, 64, 255), (780, 64, 516, 17)])
def test_layers(rt, M, mode, dims):
    x = util.normal(120, M * dims[0]).reshape(M, dims[0])
    layers, keep, src, outs = (R.GemmF32Desc * (len(dims) - 1))(), [], util.to_dev(x), []
    for l, (k, n) in enumerate(zip(dims, dims[1:])):
        w, r = util.normal(121 + l, k * n, 1.0 / np.sqrt(k)).reshape(n, k), util.normal(141 + l, M * n).reshape(M, n)
        b = util.normal(131 + l, {R.BIAS_ROW: n, R.BIAS_COL: M, R.BIAS_FULL: M * n}.get(mode, 1))
        dw, db, dr, y = util.to_dev(w), util.to_dev(b), util.to_dev(r), util.dev_empty((M, n), np.float32)
        g = layers[l]
        g.M, g.N, g.K, g.transB, g.alpha, g.beta, g.batch = M, n, k, 1, 1.0, 1.0, 1
        g.A, g.B, g.Y, g.residual, g.bias_mode, g.act = util.ptr(src), util.ptr(dw), util.ptr(y), util.ptr(dr), mode, R.ACT_RELU
        if mode != R.BIAS_NONE:
            g.C = util.ptr(db)
        keep += [src, dw, db, dr]
        b = {R.BIAS_NONE: 0.0 * b, R.BIAS_COL: b.reshape(-1, 1)}.get(mode, b.reshape(M, n) if mode == R.BIAS_FULL else b)
        outs.append((y, w.astype(np.float64), np.broadcast_to(b.astype(np.float64), (M, n)), r.astype(np.float64), k))
        src = y
    rt.set_option("f32_chain", 1)
    try:
        torch.cuda.synchronize()
        rt.call("sofie_hip_gemm_chain_f32", layers, len(layers))
        rt.sync()
    finally:
        rt.set_option("f32_chain", -1)
    inp = x.astype(np.float64)
    for y, w, b, r, k in outs:
        got = util.to_host(y).astype(np.float64)
        # every layer from the input it read: a multiply-add rounded once per k, bias and residual
        assert np.all(np.abs(got - np.maximum(inp @ w.T + b + r, 0.0)) <= (k + 3) * 2.0 ** -24 * (np.abs(inp) @ np.abs(w.T) + np.abs(b) + np.abs(r)))
        inp = got
