"""The chain kernel's layers with W stored [K,N]: up to 512 outputs k is dealt out over groups of threads, at the edges of the groups (64, 128, 256, 512 outputs),
with fewer k than groups, k that do not divide, and one, two or four rows per workgroup, the last one not filled."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 65, 131])
@pytest.mark.parametrize("dims", [(3, 1, 64, 65), (100, 128, 129, 2), (1, 256, 257, 63), (70, 512, 513, 40), (777, 33, 1030, 5)])
def test_layers(rt, M, dims):
    x = util.normal(100, M * dims[0]).reshape(M, dims[0])
    layers, keep, src, outs = (R.GemmF32Desc * (len(dims) - 1))(), [], util.to_dev(x), []
    for l, (k, n) in enumerate(zip(dims, dims[1:])):
        w, b = util.normal(101 + l, k * n, 1.0 / np.sqrt(k)).reshape(k, n), util.normal(111 + l, n)
        dw, db, y = util.to_dev(w), util.to_dev(b), util.dev_empty((M, n), np.float32)
        g = layers[l]
        g.M, g.N, g.K, g.alpha, g.beta, g.batch = M, n, k, 1.0, 1.0, 1
        g.A, g.B, g.C, g.Y, g.bias_mode, g.act = util.ptr(src), util.ptr(dw), util.ptr(db), util.ptr(y), R.BIAS_ROW, R.ACT_RELU
        keep += [src, dw, db]
        outs.append((y, w.astype(np.float64), b.astype(np.float64), k))
        src = y
    rt.set_option("f32_chain", 1)
    try:
        torch.cuda.synchronize()
        rt.call("sofie_hip_gemm_chain_f32", layers, len(layers))
        rt.sync()
    finally:
        rt.set_option("f32_chain", -1)
    inp = x.astype(np.float64)
    for y, w, b, k in outs:
        got = util.to_host(y).astype(np.float64)
        # every layer from the input it read: a multiply-add rounded once per k, and the bias
        assert np.all(np.abs(got - np.maximum(inp @ w + b, 0.0)) <= (k + 2) * 2.0 ** -24 * (np.abs(inp) @ np.abs(w) + np.abs(b)))
        inp = got
