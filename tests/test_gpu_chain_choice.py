"""Which layers of a chain share a launch, by time: against all of them together and each by itself, where the choice was a fifth to a third above the better of the two."""
import pytest
import torch

from sofie_amd import runtime as R
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M, transB, dims", [(183, 1, (128, 112, 94, 48, 3)), (202, 1, (160, 32, 104, 112, 1)), (175, 1, (6, 16, 80, 7)), (130, 1, (128, 16, 21, 48, 107)),
                                             (146, 1, (64, 48, 40, 10)), (33, 0, (16, 24, 16, 5, 5)), (20, 1, (304, 16, 32, 193))])
def test_a_fast_split_is_chosen(rt, opt, M, transB, dims):
    layers, keep, src = (R.GemmF32Desc * (len(dims) - 1))(), [], torch.randn(M * dims[0], device="cuda")
    for l, (k, n) in enumerate(zip(dims, dims[1:])):
        w, b, y = torch.randn(n * k, device="cuda"), torch.randn(n, device="cuda"), torch.empty(M * n, device="cuda")
        g = layers[l]
        g.M, g.N, g.K, g.transB, g.alpha, g.beta, g.batch = M, n, k, transB, 1.0, 1.0, 1
        g.A, g.B, g.C, g.Y, g.bias_mode, g.act = util.ptr(src), util.ptr(w), util.ptr(b), util.ptr(y), R.BIAS_ROW, R.ACT_RELU
        keep += [src, w, b, y]
        src = y
    torch.cuda.synchronize()

    def us(how):
        opt("f32_chain", how)
        best = 1e9
        for again in range(9):
            rt.timer_start()
            for _ in range(40):
                rt.call("sofie_hip_gemm_chain_f32", layers, len(layers))
            best = min(best, rt.timer_stop() * 1e3 / 40)
        return best
    us(-1)   # the card awake
    chosen, apart, together = us(-1), us(0), us(1)
    print(chosen, apart, together, flush=True)
    # (a host that does not keep up with the card lengthens the launches one by one, in every column)
    assert chosen <= 1.15 * min(apart, together)
