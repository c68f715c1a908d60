"""Performance cases of the framework: the work its users have it do, called through its public entry points.

Seven kinds of work, each over the range of sizes that occur in use:

  mlp_f32      fp32 multi-layer perceptron, one sofie_hip_gemm_chain_f32 call (what an emitted Session of Gemm + activation layers issues)
  mlp_i8       int8 quantised perceptron through Int8MLPSession
  gemm_i8      one int8 product with its requantising / dequantising store (sofie_hip_gemm_i8)
  gemm_fp8     one FP8 e4m3 product with bias and activation in its store (sofie_hip_gemm_fp8)
  cnn_i8       int8 convolutional network through Int8CNNSession
  cnn_f32      fp32 convolutional network, operator by operator as an emitted Session runs it
  encoder_f32  fp32 self-attention + feed-forward block, operator by operator as an emitted Session runs it

All work goes to one stream of the program's own, as a Session with an external stream does; inputs, weights and plans are on the
GPU before the call, and results stay there.
"""
import ctypes as C
import math

import numpy as np
import torch

from sofie_amd import Runtime
from sofie_amd import runtime as R
from sofie_amd.session import Int8CNNSession, Int8MLPSession

ACTS = {"none": R.ACT_NONE, "relu": R.ACT_RELU, "leakyrelu": R.ACT_LEAKYRELU, "sigmoid": R.ACT_SIGMOID, "tanh": R.ACT_TANH, "gelu": R.ACT_GELU}
I8_OUT = {"i8": (R.I8OUT_I8, torch.int8, 1), "f32": (R.I8OUT_F32, torch.float32, 4), "i32": (R.I8OUT_I32, torch.int32, 4)}


# ---- the cases --------------------------------------------------------------------------------------------------------

def listed():
    return [
        # the small fp32 classifier of the benchmark configurations: latency and launches count
        {"name": "mlp_f32_b64", "kind": "mlp_f32", "batch": 64, "dims": "784,128,64,10", "act": "relu", "transB": True},
        # the same kind of network over a large, ragged batch of events: throughput
        {"name": "mlp_f32_b2000", "kind": "mlp_f32", "batch": 2000, "dims": "784,1024,512,10", "act": "relu", "transB": True},
        # a few requests at a time against a wide quantised network: its weights are read for 16 rows
        {"name": "mlp_i8_b16", "kind": "mlp_i8", "batch": 16, "dims": "1024,4096,4096,1024"},
        # the headline benchmark configuration
        {"name": "mlp_i8_b1024", "kind": "mlp_i8", "batch": 1024, "dims": "1024,4096,4096,1024"},
        # an ONNX MatMulInteger of odd sizes with a run-time right operand ([K,N]), dequantised
        {"name": "gemm_i8_ragged", "kind": "gemm_i8", "M": 1537, "N": 1000, "K": 777, "out": "f32", "transB": False},
        # the benchmark configuration's large product with a requantising store
        {"name": "gemm_i8_8192", "kind": "gemm_i8", "M": 8192, "N": 8192, "K": 8192, "out": "i8", "transB": True},
        # a projection of a few rows (decode-like) in FP8
        {"name": "gemm_fp8_m50", "kind": "gemm_fp8", "M": 50, "N": 3072, "K": 1024, "act": "none", "out": "bf16"},
        # the benchmark configuration's FP8 product
        {"name": "gemm_fp8_4096", "kind": "gemm_fp8", "M": 4096, "N": 4096, "K": 4096, "act": "gelu", "out": "bf16"},
        # a small image network on a handful of small images
        {"name": "cnn_i8_b5", "kind": "cnn_i8", "batch": 5, "hw": 28, "channels": "3,16,32,64"},
        # the benchmark configuration's image network
        {"name": "cnn_i8_b256", "kind": "cnn_i8", "batch": 256, "hw": 64, "channels": "3,64,128,256,256"},
        # an fp32 image network: stem, pooling, normalisation, a residual convolution and a classifier
        {"name": "cnn_f32_b64", "kind": "cnn_f32", "batch": 64, "hw": 64, "channels": 32},
        # an fp32 attention block
        {"name": "encoder_f32_b16", "kind": "encoder_f32", "batch": 16, "seq": 128, "heads": 6, "head_dim": 64, "ff": 4},
    ]


def draw(rng):
    """One more case: a kind, and sizes over its whole range, no costlier than the listed cases of that kind."""
    kind = rng.choice(["mlp_f32", "mlp_i8", "gemm_i8", "gemm_fp8", "cnn_i8", "cnn_f32", "encoder_f32"])
    most = max(work(c)["flops"] for c in listed() if c["kind"] == kind)
    while True:
        case = _draw_kind(kind, rng)
        if work(case)["flops"] <= most:
            return case


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A matrix extent: a third multiples of 128, a third multiples of 16, a third whatever comes."""
    n, to = _log_int(rng, lo, hi), rng.choice([128, 16, 1])
    return max(to, (n + to // 2) // to * to)


def _draw_kind(kind, rng):
    if kind == "mlp_f32":
        dims = [_width(rng, 16, 2048) for _ in range(rng.randint(2, 4))] + [_log_int(rng, 1, 256)]
        return {"kind": kind, "batch": _log_int(rng, 1, 4096), "dims": ",".join(map(str, dims)), "act": rng.choice(["relu", "leakyrelu", "sigmoid", "tanh", "gelu"]),
                "transB": rng.random() < 0.5}
    if kind == "mlp_i8":
        dims = [_width(rng, 32, 4096) for _ in range(rng.randint(3, 5))]
        return {"kind": kind, "batch": _log_int(rng, 1, 4096), "dims": ",".join(map(str, dims))}
    if kind == "gemm_i8":
        return {"kind": kind, "M": _width(rng, 1, 8192), "N": _width(rng, 32, 8192), "K": _width(rng, 32, 8192), "out": rng.choice(["i8", "f32", "i32"]),
                "transB": rng.random() < 0.7}
    if kind == "gemm_fp8":
        return {"kind": kind, "M": _width(rng, 1, 4096), "N": _width(rng, 32, 4096), "K": _width(rng, 32, 4096), "act": rng.choice(["none", "relu", "gelu"]),
                "out": rng.choice(["bf16", "f32"])}
    if kind == "cnn_i8":
        channels = [rng.choice([1, 3])] + sorted(rng.choice([16, 24, 32, 64, 64, 128, 256]) for _ in range(rng.randint(2, 4)))
        return {"kind": kind, "batch": _log_int(rng, 1, 256), "hw": rng.randint(8, 64), "channels": ",".join(map(str, channels))}
    if kind == "cnn_f32":
        return {"kind": kind, "batch": _log_int(rng, 1, 64), "hw": rng.randint(12, 96), "channels": _log_int(rng, 8, 48)}
    return {"kind": kind, "batch": _log_int(rng, 1, 16), "seq": _log_int(rng, 8, 512), "heads": rng.randint(1, 12), "head_dim": rng.choice([16, 24, 32, 48, 64]),
            "ff": rng.choice([2, 4])}


def work(case):
    """Bytes and operations of one pass: every input, weight and result once, intermediates not at all; no padding, no column matrix."""
    k = case["kind"]
    if k in ("mlp_f32", "mlp_i8"):
        d, b = _dims(case["dims"]), case["batch"]
        products = sum(i * o for i, o in zip(d, d[1:]))
        if k == "mlp_i8":
            return {"bytes": 4 * b * (d[0] + d[-1]) + products, "flops": 2 * b * products}
        return {"bytes": 4 * (b * sum(d) + products + sum(d[1:])), "flops": 2 * b * products}   # every layer's output is a result
    if k in ("gemm_i8", "gemm_fp8"):
        m, n, kk = case["M"], case["N"], case["K"]
        so = I8_OUT[case["out"]][2] if k == "gemm_i8" else (2 if case["out"] == "bf16" else 4)
        return {"bytes": m * kk + n * kk + so * m * n + (8 if k == "gemm_i8" else 4) * n, "flops": 2 * m * n * kk}
    if k == "cnn_i8":
        c, b, px = _dims(case["channels"]), case["batch"], case["hw"] ** 2
        weights = sum(9 * i * o for i, o in zip(c, c[1:]))
        return {"bytes": 4 * b * c[0] * px + weights + 40 * (c[-1] + b), "flops": 2 * b * (px * weights + 10 * c[-1])}
    if k == "cnn_f32":
        b, hw, c = case["batch"], case["hw"], case["channels"]
        px = ((hw - 1) // 2 + 1) ** 2
        weights = 27 * c + 18 * c * c + 36 * c * c + 20 * c
        return {"bytes": 4 * (3 * b * hw * hw + weights + 10 * b), "flops": 2 * b * (hw * hw * 27 * c + px * 54 * c * c + 20 * c)}
    b, s, dim = case["batch"], case["seq"], case["heads"] * case["head_dim"]
    weights = (4 + 2 * case["ff"]) * dim * dim
    return {"bytes": 4 * (2 * b * s * dim + weights), "flops": 2 * b * s * (weights + 2 * s * dim)}


def tolerance(case):
    k = case["kind"]
    if k in ("mlp_i8", "gemm_i8"):
        return "exact"          # integer accumulation, and the same fp32 operations in the same order behind it
    if k == "gemm_fp8":
        # products accumulated in fp32 in the matrix cores' own order; a bf16 result may round to the neighbouring value
        return {"rel": 3e-3, "max": 1.2e-2} if case["out"] == "bf16" else {"rel": 1e-4, "max": 4e-3}
    return {"rel": 1e-5}        # fp32 sums in another order


# ---- one pass ---------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    return {"run": _PREPARE[case["kind"]](case, _Maker(seed))}


def run(state):
    return state["run"]()


_STREAM = []


def _runtime():
    """A context on the program's stream (one stream for all of them)."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return Runtime(0, external_stream=C.c_void_p(_STREAM[0].cuda_stream))


def _dims(text):
    return [int(v) for v in text.split(",")]


def _p(t):
    return C.c_void_p(t.data_ptr())


class _Maker:
    """Tensors on the GPU from a seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, sigma=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * sigma

    def uniform(self, shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def int8(self, shape):
        return torch.randint(-127, 128, shape, generator=self.g, device="cuda", dtype=torch.int8)

    def int32(self, shape, most):
        return torch.randint(-most, most + 1, shape, generator=self.g, device="cuda", dtype=torch.int32)


class _SessionOutput:
    """A Session's output region as an array other libraries can view; the view keeps the Session (which owns the memory) alive."""

    def __init__(self, session, shape):
        self.session = session
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (session.y_ptr.value, False), "version": 2, "strides": None}


def _output(session, shape):
    return torch.as_tensor(_SessionOutput(session, shape), device="cuda")


def _prepare_mlp_f32(case, make):
    rt, d, batch = _runtime(), _dims(case["dims"]), case["batch"]
    x = make.uniform((batch, d[0]))
    layers, keep, outs, src = (R.GemmF32Desc * (len(d) - 1))(), [x], [], x
    for l, (k, n) in enumerate(zip(d, d[1:])):
        w = make.normal((n, k) if case["transB"] else (k, n), 1.0 / math.sqrt(k))
        b, y = make.normal((n,), 0.1), torch.empty((batch, n), device="cuda")
        g = layers[l]
        g.M, g.N, g.K, g.transB, g.alpha, g.beta, g.batch = batch, n, k, int(case["transB"]), 1.0, 1.0, 1
        g.A, g.B, g.C, g.Y, g.bias_mode = _p(src), _p(w), _p(b), _p(y), R.BIAS_ROW
        g.act, g.act_alpha = (ACTS[case["act"]], 0.01) if l < len(d) - 2 else (R.ACT_NONE, 0.0)
        keep += [w, b]
        outs.append(y)
        src = y

    def one(keep=keep):
        rt.call("sofie_hip_gemm_chain_f32", layers, len(layers))
        return outs
    return one


def _prepare_mlp_i8(case, make):
    rt, d, batch = _runtime(), _dims(case["dims"]), case["batch"]
    x = make.normal((batch, d[0]))
    weights = [make.int8((k, n)).cpu().numpy() for k, n in zip(d, d[1:])]
    w_scale, in_scales, rms = np.float32(1.0 / 127.0), [np.float32(5.0 / 127.0)], 1.0
    for k in d[1:-1]:
        std = math.sqrt(d[len(in_scales) - 1]) * 0.577 * rms     # weights uniform on [-1, 1]; activations calibrated to four sigma
        in_scales.append(np.float32(4.0 * std / 127.0))
        rms = std / math.sqrt(2.0)
    s = Int8MLPSession(rt, weights, [w_scale] * len(weights), in_scales, batch)
    host_x = x.cpu().numpy()
    s.upload_input(host_x)
    rt.sync()
    y = _output(s, (batch, d[-1]))

    def one():
        s.infer_nosync()
        return y
    return one


def _prepare_gemm_i8(case, make):
    rt, m, n, k = _runtime(), case["M"], case["N"], case["K"]
    code, dtype, _ = I8_OUT[case["out"]]
    a, b, bias = make.int8((m, k)), make.int8((n, k) if case["transB"] else (k, n)), make.int32((n,), 1 << 15)
    scale, y = make.uniform((n,), 0.5, 1.5) / (127.0 * math.sqrt(k)), torch.empty((m, n), dtype=dtype, device="cuda")
    g = R.GemmI8Desc()
    g.M, g.N, g.K, g.transB = m, n, k, int(case["transB"])
    g.A, g.B, g.bias, g.scale, g.Y = _p(a), _p(b), _p(bias), _p(scale), _p(y)
    g.scale_scalar, g.q_scale, g.out, g.relu_out = 1.0, 1.0, code, int(case["out"] == "i8")
    room = rt.lib.sofie_hip_gemm_i8_workspace(C.byref(g))
    ws = torch.empty((max(room, 256),), dtype=torch.int8, device="cuda")
    g.workspace, g.workspace_bytes = _p(ws), room

    def one(keep=(a, b, bias, scale, ws)):
        rt.call("sofie_hip_gemm_i8", C.byref(g))
        return y
    return one


def _prepare_gemm_fp8(case, make):
    rt, m, n, k = _runtime(), case["M"], case["N"], case["K"]

    def operand(rows):
        x = make.normal((rows, k))
        s = float(x.abs().max()) / 448.0
        return (x / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8), s
    (a, sa), (b, sb) = operand(m), operand(n)
    bias, bf16 = make.normal((n,)), case["out"] == "bf16"
    y = torch.empty((m, n), dtype=torch.bfloat16 if bf16 else torch.float32, device="cuda")
    g = R.GemmFp8Desc()
    g.M, g.N, g.K, g.transB, g.scale = m, n, k, 1, sa * sb
    g.A, g.B, g.bias, g.Y = _p(a), _p(b), _p(bias), _p(y)
    g.act, g.out = ACTS[case["act"]], R.F8OUT_BF16 if bf16 else R.F8OUT_F32

    def one(keep=(a, b, bias)):
        rt.call("sofie_hip_gemm_fp8", C.byref(g))
        return y
    return one


def _prepare_cnn_i8(case, make):
    rt, c, batch, hw = _runtime(), _dims(case["channels"]), case["batch"], case["hw"]
    convs = []
    for cin, cout in zip(c, c[1:]):
        # accumulators have a spread of about 73 * 40 * sqrt(9 cin); the scale brings them back to a spread of about 40
        scale = make.uniform((cout,), 0.5, 1.5) * (0.0138 / math.sqrt(9 * cin))
        convs.append(dict(W=make.int8((cout, cin, 3, 3)).cpu().numpy(), bias=make.int32((cout,), 3000).cpu().numpy(), scale=scale.cpu().numpy(),
                          pads=(1, 1, 1, 1), strides=(1, 1), dils=(1, 1)))
    fc_w, fc_b = make.normal((c[-1], 10), 0.05).cpu().numpy(), make.normal((10,), 0.1).cpu().numpy()
    s = Int8CNNSession(rt, batch, (c[0], hw, hw), np.float32(1.0 / 127.0), convs, np.float32(0.05), fc_w, fc_b)
    host_x = make.uniform((batch, c[0], hw, hw)).cpu().numpy()
    s.upload_input(host_x)
    rt.sync()
    y = _output(s, (batch, 10))

    def one():
        s.infer_nosync()
        return y
    return one


def _in_order(rt, calls, outputs, keep):
    """A pass that issues `calls` one after the other; `keep` holds the memory they point to."""
    def one(keep=keep):
        for call in calls:
            rt.call(*call)
        return outputs
    return one


def _gemm(a, b, y, m, n, k, bias=None, transB=0, alpha=1.0, act=R.ACT_NONE, batch=1, residual=None):
    g = R.GemmF32Desc()
    g.M, g.N, g.K, g.transB, g.alpha, g.beta, g.batch, g.act = m, n, k, transB, alpha, 1.0, batch, act
    g.A, g.B, g.Y = _p(a), _p(b), _p(y)
    if bias is not None:
        g.C, g.bias_mode = _p(bias), R.BIAS_ROW
    if residual is not None:
        g.residual = _p(residual)
    if batch > 1:
        g.strideA, g.strideB, g.strideY = m * k, n * k, m * n
    return g


def _prepare_cnn_f32(case, make):
    rt, n, hw, c = _runtime(), case["batch"], case["hw"], case["channels"]
    half = (hw - 1) // 2 + 1
    x = make.uniform((n, 3, hw, hw))

    def conv(cin, cout, h):
        d = R.ConvDesc()
        d.N, d.C, d.H, d.W, d.Cout, d.kh, d.kw, d.group, d.OH, d.OW = n, cin, h, h, cout, 3, 3, 1, h, h
        d.pad_h0 = d.pad_w0 = d.pad_h1 = d.pad_w1 = d.stride_h = d.stride_w = d.dil_h = d.dil_w = 1
        return d, make.normal((cout, cin, 3, 3), math.sqrt(2.0 / (9 * cin))), make.normal((cout,), 0.1), torch.empty((n, cout, h, h), device="cuda")
    (d1, w1, b1, y1), (d2, w2, b2, y2), (d3, w3, b3, y3) = conv(3, c, hw), conv(c, 2 * c, half), conv(2 * c, 2 * c, half)
    pool = R.PoolDesc()
    pool.planes, pool.H, pool.W, pool.OH, pool.OW, pool.kh, pool.kw = n * c, hw, hw, half, half, 3, 3
    pool.pad_h0 = pool.pad_w0 = pool.pad_h1 = pool.pad_w1 = 1
    pool.stride_h = pool.stride_w = 2
    pool.mode, pool.dynamic_divisor = R.POOL_MAX, 1
    p1, bn = torch.empty((n, c, half, half), device="cuda"), torch.empty_like(y2)
    fused, mean, beta = make.uniform((2 * c,), 0.5, 1.5), make.normal((2 * c,), 0.5), make.normal((2 * c,), 0.2)
    avg, logits, prob = (torch.empty((n, k), device="cuda") for k in (2 * c, 10, 10))
    wf, bf = make.normal((2 * c, 10), 0.3), make.normal((10,), 0.1)
    fc = _gemm(avg, wf, logits, n, 10, 2 * c, bias=bf)
    zero, none = C.c_float(0.0), None

    calls = [("sofie_hip_conv_f32", C.byref(d1), _p(x), _p(w1), _p(b1), R.ACT_RELU, zero, _p(y1), none, none),
             ("sofie_hip_pool_f32", C.byref(pool), _p(p1), _p(y1)),
             ("sofie_hip_conv_f32", C.byref(d2), _p(p1), _p(w2), _p(b2), R.ACT_NONE, zero, _p(y2), none, none),
             ("sofie_hip_batchnorm_f32", _p(bn), _p(y2), _p(fused), _p(mean), _p(beta), n, 2 * c, half * half, 1),
             ("sofie_hip_conv_f32", C.byref(d3), _p(bn), _p(w3), _p(b3), R.ACT_RELU, zero, _p(y3), none, _p(bn)),
             ("sofie_hip_global_avg_pool_f32", _p(avg), _p(y3), n * 2 * c, half * half),
             ("sofie_hip_gemm_f32", C.byref(fc)),
             ("sofie_hip_softmax_f32", _p(prob), _p(logits), n, 10, 1, 0)]
    return _in_order(rt, calls, [y3, avg, logits, prob], (x, w1, b1, w2, b2, w3, b3, p1, y1, y2, bn, fused, mean, beta, wf, bf))


def _prepare_encoder_f32(case, make):
    rt, b, s, h, d = _runtime(), case["batch"], case["seq"], case["heads"], case["head_dim"]
    t, dim, wide = b * s, h * d, case["ff"] * h * d

    def new(*shape):
        return torch.empty(shape, device="cuda")

    def linear(k, n):
        return make.normal((k, n), 1.0 / math.sqrt(k)), make.normal((n,), 0.1)
    x = make.normal((t, dim))
    g1, be1, g2, be2 = make.uniform((dim,), 0.8, 1.2), make.normal((dim,), 0.1), make.uniform((dim,), 0.8, 1.2), make.normal((dim,), 0.1)
    n1, n2, y1, y2, ctx, merged, up = new(t, dim), new(t, dim), new(t, dim), new(t, dim), new(b * h, s, d), new(t, dim), new(t, wide)
    scores, prob = new(b * h, s, s), new(b * h, s, s)
    proj, keep = [], [x, g1, be1, g2, be2]
    for _ in range(3):
        (w, bias), flat, split = linear(dim, dim), new(t, dim), new(b * h, s, d)
        proj.append((_gemm(n1, w, flat, t, dim, dim, bias=bias), flat, split))
        keep += [w, bias]
    (wo, bo), (w1, b1), (w2, b2) = linear(dim, dim), linear(dim, wide), linear(wide, dim)
    keep += [wo, bo, w1, b1, w2, b2]
    q, k, v = (split for _, _, split in proj)
    qk = _gemm(q, k, scores, s, s, d, transB=1, alpha=1.0 / math.sqrt(d), batch=b * h)
    pv = _gemm(prob, v, ctx, s, d, s, batch=b * h)
    out = _gemm(merged, wo, y1, t, dim, dim, bias=bo, residual=x)
    ff1, ff2 = _gemm(n2, w1, up, t, wide, dim, bias=b1, act=R.ACT_GELU), _gemm(up, w2, y2, t, dim, wide, bias=b2, residual=y1)
    swap = (C.c_int32 * 4)(0, 2, 1, 3)
    apart, joined = (C.c_int64 * 4)(b, s, h, d), (C.c_int64 * 4)(b, h, s, d)
    eps = C.c_float(1e-5)

    calls = [("sofie_hip_layernorm_f32", _p(n1), _p(x), _p(g1), _p(be1), t, dim, eps, None, None)]
    for g, flat, split in proj:
        calls += [("sofie_hip_gemm_f32", C.byref(g)), ("sofie_hip_transpose_f32", _p(split), _p(flat), 4, apart, swap)]
    calls += [("sofie_hip_gemm_f32", C.byref(qk)),
              ("sofie_hip_softmax_f32", _p(prob), _p(scores), b * h * s, s, 1, 0),
              ("sofie_hip_gemm_f32", C.byref(pv)),
              ("sofie_hip_transpose_f32", _p(merged), _p(ctx), 4, joined, swap),
              ("sofie_hip_gemm_f32", C.byref(out)),
              ("sofie_hip_layernorm_f32", _p(n2), _p(y1), _p(g2), _p(be2), t, dim, eps, None, None),
              ("sofie_hip_gemm_f32", C.byref(ff1)),
              ("sofie_hip_gemm_f32", C.byref(ff2))]
    return _in_order(rt, calls, [y1, y2], keep + [n1, n2, ctx, merged, up, scores, prob, proj])


_PREPARE = {"mlp_f32": _prepare_mlp_f32, "mlp_i8": _prepare_mlp_i8, "gemm_i8": _prepare_gemm_i8, "gemm_fp8": _prepare_gemm_fp8,
            "cnn_i8": _prepare_cnn_i8, "cnn_f32": _prepare_cnn_f32, "encoder_f32": _prepare_encoder_f32}
