"""The choice among the kernels of the fp32 products, by time, where batches of products that come float by float were taken to tiles of 128 x 128 although smaller ones are faster."""
import ctypes as C

import pytest
import torch

from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M, N, K, batch, transA, transB", [(693, 163, 19, 63, 0, 1), (1712, 48, 19, 124, 0, 1), (640, 223, 85, 52, 0, 1), (432, 351, 64, 54, 0, 0), (176, 1297, 32, 89, 1, 0),
                                                            (361, 256, 64, 87, 1, 0), (787, 400, 1342, 1, 1, 0)])
def test_a_fast_kernel_is_chosen(rt, opt, M, N, K, batch, transA, transB):
    """Where the costs were fitted the choice is at most 31 % above the fastest kernel, and 7 % here; it was 30 % to twice its time in the first six."""
    A, B, Y = (torch.randn(n, device="cuda") for n in (batch * M * K, batch * N * K, batch * M * N))
    g = R.GemmF32Desc()
    g.M, g.N, g.K, g.transA, g.transB, g.alpha, g.batch = M, N, K, transA, transB, 1.0, batch
    g.A, g.B, g.Y, g.strideA, g.strideB, g.strideY = util.ptr(A), util.ptr(B), util.ptr(Y), M * K, N * K, M * N
    torch.cuda.synchronize()

    def us(tile):
        opt("f32_tile", tile)
        best = 1e9
        for again in range(7):
            rt.timer_start()
            for _ in range(20):
                rt.call("sofie_hip_gemm_f32", C.byref(g))
            best = min(best, rt.timer_stop() * 1e3 / 20)
        return best
    us(0)   # the card awake
    times = {tile: us(tile) for tile in (0, 16, 32, 62, 64, 128)}
    print(times, flush=True)
    assert times[0] <= 1.2 * min(times.values())
