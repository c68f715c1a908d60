"""The longest extents of a product: what lies past them is refused before a launch (tile arithmetic would leave 32 bits)."""
import ctypes as C

import pytest

from sofie_amd import runtime as R

MOST = (1 << 31) - 256          # rows of a product: the last tile, of at most 256, ends within 32 bits


def refused(name, *args):
    room = C.create_string_buffer(4096)          # a context that no launch is made on
    lib = R.load_library()
    assert getattr(lib, name)(C.addressof(room), *args) == 1
    return lib.sofie_hip_last_error().decode()


@pytest.mark.parametrize("M, N", [(MOST + 1, 1), ((1 << 31) - 1, 1), (1, MOST + 1), (1, (1 << 31) - 1)])
@pytest.mark.parametrize("kind", [R.GemmF32Desc, R.GemmI8Desc, R.GemmFp8Desc])
def test_products_past_the_longest_are_refused(kind, M, N):
    d = kind()
    d.M, d.N, d.K, d.transB, d.A, d.B, d.Y = M, N, 1, 1, 4096, 4096, 4096
    if kind is R.GemmF32Desc:
        d.batch, d.alpha = 1, 1.0
        chain = (kind * 2)(d, d)
        chain[0].A, chain[1].A = 8192, 4096
        assert "M or N too long" in refused("sofie_hip_gemm_chain_f32", chain, 2)
    name = {R.GemmF32Desc: "sofie_hip_gemm_f32", R.GemmI8Desc: "sofie_hip_gemm_i8", R.GemmFp8Desc: "sofie_hip_gemm_fp8"}[kind]
    assert "M or N too long" in refused(name, C.byref(d))


def test_convolutions_past_the_longest_are_refused():
    d = R.ConvDesc()
    d.N = d.C = d.Cout = d.kh = d.kw = d.stride_h = d.stride_w = d.dil_h = d.dil_w = d.group = 1
    d.W = d.OW = 64
    d.H = d.OH = MOST // 64 + 1
    assert MOST < d.OH * d.OW < 1 << 31
    for residual in (None, 4096):
        assert "too many output pixels" in refused("sofie_hip_conv_f32", C.byref(d), 4096, 4096, None, 0, 0.0, 4096, None, residual)
    a = R.ConvI8Args()
    a.X = a.W = a.Y = a.scale = 4096
    a.out, a.w_is_packed = R.I8OUT_I8, 1
    assert "too many output pixels" in refused("sofie_hip_conv_i8", C.byref(d), C.byref(a))


def test_re_layouts_past_the_longest_are_refused():
    assert "too many rows" in refused("sofie_hip_transpose_i8", 4096, 8192, (1 << 31) - 1, 1, 0, 0)
    assert "too many rows" in refused("sofie_hip_transpose_i8", 4096, 8192, 65535 * 64 + 1, 16, 0, 0)
