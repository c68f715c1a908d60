"""Chains in one launch whose layers differ in how W is stored: [K,N] alone (the kernel without the loop over rows of W), rows of 16-byte pieces between layers of the other forms, rows
that are padded, by whole pieces and not, and W that does not start on 16 bytes.  Every layer is held to the input that it read."""
import ctypes as C

import numpy as np
import pytest
import torch

from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu
# storage of a layer's W: transposed or not, floats behind its rows, floats before it
COLUMNS, PADDED_COLUMNS, ROWS, WHOLE_PIECES, OTHER_ROWS, OFF = (0, 0, 0), (0, 3, 1), (1, 0, 0), (1, 8, 0), (1, 3, 0), (1, 4, 1)


@pytest.mark.parametrize("M", [3, 65, 130])
@pytest.mark.parametrize("dims", [(64, 257, 60, 5), (132, 128, 516, 17), (4, 64, 4, 130)])
@pytest.mark.parametrize("forms", [(COLUMNS, COLUMNS, COLUMNS), (PADDED_COLUMNS, COLUMNS, PADDED_COLUMNS), (COLUMNS, ROWS, COLUMNS), (WHOLE_PIECES, COLUMNS, WHOLE_PIECES),
                                   (OTHER_ROWS, OTHER_ROWS, OFF), (OFF, WHOLE_PIECES, OTHER_ROWS), (ROWS, OFF, COLUMNS)])
def test_forms_of_weights(rt, opt, M, dims, forms):
    seed = 300 + M + sum(dims)
    x = util.normal(seed, M * dims[0]).reshape(M, dims[0])
    layers, keep, src, outs = (R.GemmF32Desc * 3)(), [], util.to_dev(x), []
    for l, (k, n, (transposed, pad, before)) in enumerate(zip(dims, dims[1:], forms)):
        rows, cols = (n, k) if transposed else (k, n)
        room = np.full(before + rows * (cols + pad) + 8, np.nan, dtype=np.float32)   # what pads W is never used
        w = util.normal(seed + 10 + l, rows * cols, 1.0 / np.sqrt(k)).reshape(rows, cols)
        room[before : before + rows * (cols + pad)].reshape(rows, cols + pad)[:, :cols] = w
        b = util.normal(seed + 20 + l, n)
        dw, db, y = util.to_dev(room), util.to_dev(b), util.dev_empty((M, n), np.float32)
        g = layers[l]
        g.M, g.N, g.K, g.transB, g.ldb, g.alpha, g.beta, g.batch = M, n, k, transposed, cols + pad, 1.0, 1.0, 1
        g.A, g.B, g.C, g.Y, g.bias_mode, g.act = util.ptr(src), C.c_void_p(dw.data_ptr() + 4 * before), util.ptr(db), util.ptr(y), R.BIAS_ROW, R.ACT_RELU
        keep += [src, dw, db]
        outs.append((y, (w.T if transposed else w).astype(np.float64), b.astype(np.float64), k))
        src = y
    torch.cuda.synchronize()
    opt("f32_chain", 1)
    rt.call("sofie_hip_gemm_chain_f32", layers, 3)
    rt.sync()
    inp = x.astype(np.float64)
    for y, w, b, k in outs:
        got = util.to_host(y).astype(np.float64)
        # a multiply-add rounded once per k, the sums of groups added up, the bias
        assert np.all(np.abs(got - np.maximum(inp @ w + b, 0.0)) <= (k + 20) * 2.0 ** -24 * (np.abs(inp) @ np.abs(w) + np.abs(b)))
        inp = got
