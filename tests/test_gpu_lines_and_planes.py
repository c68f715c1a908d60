"""The register-resident line kernels (Softmax, LayerNormalization), the planes (BatchNormalization, GlobalAveragePool) and the axis-folding
Transpose at the sizes where their loops, lane groups and vector paths end, each against its definition in float64 or numpy's own result."""
import ctypes as C

import numpy as np
import pytest

from tests import util

pytestmark = pytest.mark.gpu

# one lane, a full group, one more than a group, the last length in registers and the first beyond, for scalars and for vectors of four
LINES = [1, 2, 3, 4, 5, 8, 63, 64, 65, 68, 128, 252, 255, 256, 257, 260, 512, 516, 1000, 1023, 1024, 1025, 1028]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n", LINES)
def test_lines(rt, n, offset):
    rows = 131 if n <= 64 else 7      # a last wave that is not full
    X = (2 * util.normal(7000 + n, rows * n)).reshape(rows, n).astype(np.float32)
    g, b = util.normal(7001, n), util.normal(7002, n)
    dX, dY, dG, dB = util.to_dev(np.concatenate([np.zeros(offset, np.float32), X.ravel()])), util.to_dev(np.full(rows * n + 8, 7.0, np.float32)), util.to_dev(g), util.to_dev(b)
    x = C.c_void_p(util.ptr(dX).value + 4 * offset)
    x64 = X.astype(np.float64)
    e = np.exp(x64 - x64.max(1, keepdims=True))
    for log in (0, 1):
        rt.call("sofie_hip_softmax_f32", util.ptr(dY), x, rows, n, 1, log)
        rt.sync()
        got, want = util.to_host(dY), e / e.sum(1, keepdims=True)
        assert np.all(got[rows * n:] == 7.0)
        if log:
            assert np.allclose(got[:rows * n].reshape(rows, n), np.log(want), rtol=1e-6, atol=4e-6)
        else:
            assert np.allclose(got[:rows * n].reshape(rows, n), want, rtol=3e-6, atol=0)
    rt.call("sofie_hip_layernorm_f32", util.ptr(dY), x, util.ptr(dG), util.ptr(dB), rows, n, C.c_float(1e-5), None, None)
    rt.sync()
    got = util.to_host(dY)
    want = (x64 - x64.mean(1, keepdims=True)) / np.sqrt(x64.var(1, keepdims=True) + 1e-5) * g + b
    assert np.all(got[rows * n:] == 7.0) and np.allclose(got[:rows * n].reshape(rows, n), want, rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("n,c,hw", [(1, 1, 1), (2, 3, 4), (3, 5, 255), (1, 2, 256), (2, 7, 1020), (5, 3, 1024), (2, 2, 1028), (1, 3, 4100)])
def test_planes(rt, n, c, hw):
    X = util.normal(7100, n * c * hw).reshape(n, c, hw)
    f, m, b = util.normal(7101, c), util.normal(7102, c), util.normal(7103, c)
    dX, dY, dA, dF, dM, dB = util.to_dev(X), util.dev_empty(X.shape, np.float32), util.dev_empty((n, c), np.float32), util.to_dev(f), util.to_dev(m), util.to_dev(b)
    rt.call("sofie_hip_batchnorm_f32", util.ptr(dY), util.ptr(dX), util.ptr(dF), util.ptr(dM), util.ptr(dB), n, c, hw, 1)
    rt.call("sofie_hip_global_avg_pool_f32", util.ptr(dA), util.ptr(dX), n * c, hw)
    rt.sync()
    want = np.maximum((X - m[:, None]) * f[:, None] + b[:, None], np.float32(0))
    assert np.array_equal(util.to_host(dY), want)
    assert np.allclose(util.to_host(dA), X.astype(np.float64).mean(2), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("shape,perm", [((2, 5, 3, 8), (0, 2, 1, 3)), ((2, 5, 3, 7), (0, 2, 1, 3)), ((4, 6), (1, 0)), ((3, 4, 8), (0, 1, 2)), ((1, 1), (1, 0)),
                                        ((2, 1, 3, 1, 4), (3, 2, 0, 1, 4)), ((2, 3, 4, 5, 2, 4), (5, 4, 3, 2, 1, 0)), ((300, 7, 260), (1, 0, 2))])
def test_transpose_axes(rt, shape, perm):
    X = util.normal(7200, int(np.prod(shape))).reshape(shape)
    dX, dY = util.to_dev(X), util.dev_empty((X.size,), np.float32)
    rank = len(shape)
    rt.call("sofie_hip_transpose_f32", util.ptr(dY), util.ptr(dX), rank, (C.c_int64 * rank)(*shape), (C.c_int32 * rank)(*perm))
    rt.sync()
    assert np.array_equal(util.to_host(dY), np.transpose(X, perm).ravel())
