"""A Session reads its scales and descriptors at each pass: what a program changes after construction holds from the next pass on."""
import ctypes as C

import numpy as np
import pytest

from sofie_amd import runtime as R
from sofie_amd.session import Int8CNNSession, Int8MLPSession


class _Runtime:
    """Notes the calls instead of making them."""
    ctx = None

    def __init__(self):
        self.lib, self.made = self, []
        self.real = R.load_library()

    def __getattr__(self, name):
        return getattr(self.real, name)

    def sofie_hip_arena_ptr(self, ctx, offset):
        return 4096 + offset.value

    def call(self, name, *args):
        self.made.append((name, [a._obj if type(a) is type(C.byref(C.c_int())) else getattr(a, "value", a) for a in args]))

    def sync(self):
        pass

    def one_pass(self, session):
        self.made.clear()
        session.infer_nosync()
        return list(self.made)


def test_mlp_attributes_hold_from_the_next_pass():
    rt = _Runtime()
    s = Int8MLPSession(rt, [np.ones((32, 48), np.int8), np.ones((48, 16), np.int8)], [1.0, 1.0], [0.5, 0.25], 3)
    first = rt.one_pass(s)
    assert [c[0] for c in first] == ["sofie_hip_quantize_linear"] + ["sofie_hip_gemm_i8"] * 2
    assert first[0][1] == [s.p(s.off_xq).value, s.x_ptr.value, 96, 0.5] and first[1][1][0] is s.descs[0]
    s.in_scales[0] = np.float32(0.125)
    s.descs[1] = R.GemmI8Desc()
    second = rt.one_pass(s)
    assert second[0][1][3] == 0.125 and second[1] == first[1] and second[2][1][0] is s.descs[1]


@pytest.mark.parametrize("pool_in_conv", [False, True])
def test_cnn_attributes_hold_from_the_next_pass(pool_in_conv):
    rt = _Runtime()
    convs = [dict(W=np.ones((64, cin, 3, 3), np.int8), bias=np.zeros(64, np.int32), scale=np.ones(64, np.float32), pads=(1, 1, 1, 1)) for cin in (3, 64)]
    s = Int8CNNSession(rt, 2, (3, 16, 16), 0.5, convs, 0.25, np.ones((64, 10), np.float32), np.zeros(10, np.float32), pool_in_conv)
    assert s.pool_in_conv == pool_in_conv
    first = rt.one_pass(s)
    average = "sofie_hip_plane_sums_to_average" if pool_in_conv else "sofie_hip_global_avg_pool_i8"
    assert [c[0] for c in first] == ["sofie_hip_quantize_linear"] + ["sofie_hip_fill_zero"] * pool_in_conv + ["sofie_hip_conv_i8"] * 2 + [average, "sofie_hip_gemm_f32"]
    assert first[0][1] == [s.p(s.off_xq).value, s.x_ptr.value, 2 * 3 * 256, 0.5] and first[-2][1][-1] == 0.25
    s.in_scale, s.last_scale, s.fc, s.conv_args[1] = np.float32(0.125), np.float32(2.0), R.GemmF32Desc(), R.ConvI8Args()
    second = rt.one_pass(s)
    assert second[0][1][3] == 0.125 and second[-2][1][-1] == 2.0 and second[-1][1][0] is s.fc and second[-3][1][1] is s.conv_args[1]
