"""Long extents: lists of tiles of 2^32 threads and more, rows up to the longest that is taken.  One column and a reduction of a few
elements keep the arithmetic small; every result is compared, on the GPU, with torch's of the same operation."""
import ctypes as C

import pytest
import torch

from sofie_amd import runtime as R

pytestmark = pytest.mark.gpu

MOST = (1 << 31) - 256


def p(t):
    return C.c_void_p(t.data_ptr())


@pytest.fixture(autouse=True)
def memory():
    yield
    torch.cuda.empty_cache()


# 32 x 32 tiles of 256 threads: 2^32 threads from 2^29 rows on; 16 x 16 tiles of 512: from 2^27 on
@pytest.mark.parametrize("M, K, transA, tile", [((1 << 29) + 5, 1, 0, 0), (MOST, 1, 0, 0), ((1 << 27) + 77, 0, 0, 0), ((1 << 27) + 77, 3, 1, 16), (MOST, 1, 0, 16)])
def test_fp32_products_of_many_rows(rt, opt, M, K, transA, tile):
    print("gemm_f32", M, K, transA, tile, flush=True)
    A = torch.rand((K, M) if transA else (M, K), device="cuda")
    b, c, y = torch.rand(max(K, 1), device="cuda"), torch.rand(1, device="cuda"), torch.empty(M, device="cuda")
    d = R.GemmF32Desc()
    d.M, d.N, d.K, d.transA, d.transB, d.alpha, d.beta, d.batch, d.bias_mode = M, 1, K, transA, 1, 1.0, 1.0, 1, R.BIAS_ROW
    d.A, d.B, d.C, d.Y = p(A), p(b), p(c), p(y)
    torch.cuda.synchronize()
    opt("f32_tile", tile)
    rt.call("sofie_hip_gemm_f32", C.byref(d))
    rt.sync()
    want = c.expand(M).clone()
    for k in range(K):
        want += (A[k] if transA else A[:, k]) * b[k]
    # K + 1 roundings of values below K + 1, in either order
    assert float(want.sub_(y).abs_().max()) <= 4 * (K + 1) ** 2 * 2.0 ** -24


# rows of less than 16 bytes go to the direct kernel: 2^32 threads from 2^31 results on
@pytest.mark.parametrize("kind", ["int8", "fp8"])
def test_narrow_8_bit_products_of_many_rows(rt, kind):
    M, N, K = (1 << 26) + 9, 32, 2
    print("gemm", kind, M, N, K, flush=True)
    if kind == "int8":
        A, B, y = torch.randint(-7, 8, (M, K), device="cuda", dtype=torch.int8), torch.randint(-7, 8, (N, K), device="cuda", dtype=torch.int8), torch.empty((M, N), dtype=torch.int8, device="cuda")
        d, scale, values = R.GemmI8Desc(), torch.ones(N, device="cuda"), lambda t: t
        d.scale, d.scale_scalar, d.q_scale, d.out = p(scale), 1.0, 1.0, R.I8OUT_I8
    else:
        codes = torch.tensor([0x00, 0x38, 0x40, 0xb8], dtype=torch.uint8, device="cuda")                # 0, 1, 2, -1 in e4m3
        A, B = (codes[torch.randint(0, 4, (n, K), device="cuda", dtype=torch.uint8).long()] for n in (M, N))
        y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
        d, values = R.GemmFp8Desc(), lambda t: t.view(torch.float8_e4m3fn).to(torch.bfloat16)
        d.scale, d.out = 1.0, R.F8OUT_BF16
    d.M, d.N, d.K, d.transB, d.A, d.B, d.Y = M, N, K, 1, p(A), p(B), p(y)
    torch.cuda.synchronize()
    rt.call("sofie_hip_gemm_i8" if kind == "int8" else "sofie_hip_gemm_fp8", C.byref(d))
    rt.sync()
    a, b = values(A), values(B)
    for n in range(N):          # small whole numbers: exact in either type
        assert torch.equal(y[:, n], a[:, 0] * b[n, 0] + a[:, 1] * b[n, 1]), n


@pytest.mark.parametrize("images, hw, kernel, tile", [(1, (1 << 14, (1 << 13) + 1), 1, 16), ((1 << 29) // 3844 + 2, (62, 62), 3, 3032)])
def test_fp32_convolutions_of_many_pixels(rt, opt, images, hw, kernel, tile):
    print("conv_f32", images, hw, kernel, tile, flush=True)
    d = R.ConvDesc()
    d.N, d.C, d.Cout, d.group, d.H, d.OH, d.W, d.OW, d.kh, d.kw = images, 1, 1, 1, hw[0], hw[0], hw[1], hw[1], kernel, kernel
    d.pad_h0 = d.pad_w0 = d.pad_h1 = d.pad_w1 = kernel // 2
    d.stride_h = d.stride_w = d.dil_h = d.dil_w = 1
    x, y = torch.rand((images,) + hw, device="cuda"), torch.empty((images,) + hw, device="cuda")
    w = torch.rand((kernel, kernel), device="cuda")
    torch.cuda.synchronize()
    opt("f32_tile", tile)
    rt.call("sofie_hip_conv_f32", C.byref(d), p(x), p(w), None, R.ACT_NONE, C.c_float(0), p(y), None, None)
    rt.sync()
    want, h = torch.zeros_like(x), kernel // 2
    for i in range(kernel):
        for j in range(kernel):
            rows, columns = slice(max(0, h - i), hw[0] - max(0, i - h)), slice(max(0, h - j), hw[1] - max(0, j - h))
            want[:, rows, columns] += w[i, j] * x[:, max(0, i - h):hw[0] - max(0, h - i), max(0, j - h):hw[1] - max(0, h - j)]
    # nine products of values below one, added in either order
    assert float(want.sub_(y).abs_().max()) <= 2 * 9 * 9 * 2.0 ** -24


@pytest.mark.parametrize("Cout", [3, 64])
def test_int8_convolution_of_a_tall_image(rt, Cout):
    """More rows than 2^24: the unused places of a window kernel's reduction still lie outside the image."""
    H, W = (1 << 24) + 40, 8
    print("conv_i8", H, W, Cout, flush=True)
    x, w = torch.randint(-3, 4, (H, W), device="cuda", dtype=torch.int8), torch.randint(-2, 3, (Cout, 3, 3), device="cuda", dtype=torch.int8)
    y, scale = torch.empty((H, W, Cout), device="cuda", dtype=torch.int8), torch.ones(Cout, device="cuda")
    d, a = R.ConvDesc(), R.ConvI8Args()
    d.N, d.C, d.Cout, d.group, d.H, d.OH, d.W, d.OW, d.kh, d.kw = 1, 1, Cout, 1, H, H, W, W, 3, 3
    d.pad_h0 = d.pad_w0 = d.pad_h1 = d.pad_w1 = d.stride_h = d.stride_w = d.dil_h = d.dil_w = 1
    packed = torch.zeros(rt.lib.sofie_hip_conv_weight_i8_packed_bytes(C.byref(d)), device="cuda", dtype=torch.int8)
    torch.cuda.synchronize()
    rt.call("sofie_hip_pack_conv_weight_i8", C.byref(d), p(packed), p(w))
    a.X, a.W, a.scale, a.Y, a.out, a.w_is_packed = p(x), p(packed), p(scale), p(y), R.I8OUT_I8, 1
    a.x_layout, a.y_layout = R.LAYOUT_NCHW, R.LAYOUT_NHWC
    rt.call("sofie_hip_conv_i8", C.byref(d), C.byref(a))
    rt.sync()
    padded = torch.zeros((H + 2, W + 2), device="cuda", dtype=torch.int8)
    padded[1:-1, 1:-1] = x
    for c in (0, 1, Cout - 1):          # sums of at most 54: exact in 8 bits
        want = sum(w[c, i, j] * padded[i:i + H, j:j + W] for i in range(3) for j in range(3))
        assert torch.equal(y[:, :, c], want), c
