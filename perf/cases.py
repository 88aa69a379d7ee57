"""The work this library is timed on: one pass of each operator family over the range of sizes, data types and options
it is used with, through the operators' own surface (MakeArgumentPointer / MakeInvokerPointer().Run).

`listed()` names one case per way of using the library; `draw(rng)` gives another case of the same ranges. Every case is
a dict of plain values with a `kind`:

    gemm       DeviceGemm{Int8,F16,BF16}; int8 with the rounded requant-ReLU-requant epilogue
    conv       DeviceConv2dFwd{Int8,F16} / DeviceConv2dFwdBiasActivationF16 / DeviceConvNdFwd{Int8,F16}
    gemm_gemm  DeviceBatchedGemmGemmF16, or with `softmax` DeviceBatchedGemmSoftmaxGemmF16 (attention), `mask`: causal

`prepare` builds what a program holds before the call (operands, operator, argument, the workspace that
GetWorkSpaceSize asks for); `run` is one Run() of the invoker on the current stream.
"""
import math

import torch

import composable_kernel_amd as ck


def _gemm(name, dtype, M, N, K, layout="mk_nk"):
    return {"name": name, "kind": "gemm", "dtype": dtype, "M": M, "N": N, "K": K, "layout": layout}


def _conv(name, dtype, N, C, K, hw, f, stride=1, pad=0, dil=1, ndim=2, fused=""):
    return {"name": name, "kind": "conv", "dtype": dtype, "ndim": ndim, "N": N, "C": C, "K": K, "hw": hw, "f": f,
            "stride": stride, "pad": pad, "dil": dil, "fused": fused}


def _gemm_gemm(name, G, M, N, K, O, softmax=False, mask=False):
    return {"name": name, "kind": "gemm_gemm", "dtype": "f16", "G": G, "M": M, "N": N, "K": K, "O": O,
            "softmax": softmax, "mask": mask}


def listed():
    return [
        # the smallest call: a fused pair of batched GEMMs of a few microseconds (latency and launch count)
        _gemm_gemm("gemm_gemm_b64_512", 64, 512, 512, 64, 64),
        # one token through a quantised linear layer (decode of a single sequence): the weights are read once
        _gemm("i8_m1_n11008_k4096", "i8", 1, 11008, 4096),
        # 128 tokens (batched decode, a short prompt) through the layer with the long reduction
        _gemm("i8_m128_n4096_k11008", "i8", 128, 4096, 11008),
        # a long prompt through the quantised layer: the largest of the integer GEMMs
        _gemm("i8_m4096_n11008_k4096", "i8", 4096, 11008, 4096),
        # the square fp16 GEMM the library is quoted on
        _gemm("f16_4096", "f16", 4096, 4096, 4096),
        # bf16 activations against a row-major weight matrix (x @ W as frameworks store W)
        _gemm("bf16_kn_m2048_n8192_k2048", "bf16", 2048, 8192, 2048, "mk_kn"),
        # sizes that are no multiple of anything: the padded instances (KPadding / MNKPadding)
        _gemm("f16_ragged_m2001_n1003_k1025", "f16", 2001, 1003, 1025),
        # the 3x3 stride-2 layer the conv operators are quoted on, with bias + ReLU
        _conv("conv_f16_n128_c192_k256_3x3_71_s2", "f16", 128, 192, 256, 71, 3, 2, 1, fused="bias_relu"),
        # a quantised mid-network 3x3 layer at an inference batch
        _conv("conv_i8_n32_c256_k256_3x3_14", "i8", 32, 256, 256, 14, 3, 1, 1),
        # the first layer of an image network: three input channels (the OddC instances)
        _conv("conv_f16_n64_c3_k32_3x3_224_s2", "f16", 64, 3, 32, 224, 3, 2, 1, fused="bias_relu"),
        # three spatial dimensions
        _conv("conv3d_f16_n16_c64_k64_3x3x3_32", "f16", 16, 64, 64, 32, 3, 1, 1, ndim=3),
        # causal attention over a long sequence, 64 batch-heads
        _gemm_gemm("attention_causal_b64_4096", 64, 4096, 4096, 64, 64, softmax=True, mask=True),
    ]


# ------------------------------------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi, step=1):
    """A whole multiple of `step` in [lo, hi], uniform in its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi // step * step, max(-(-lo // step) * step, int(round(v / step)) * step))


def _draw_one(rng):
    family = rng.choice(["decode", "tokens", "large", "layout", "ragged", "conv", "conv", "odd_conv", "conv3d",
                         "gemm_gemm", "attention", "attention"])
    if family == "decode":    # a few rows against a weight matrix
        return _gemm("", rng.choice(["i8", "i8", "f16", "bf16"]), _log(rng, 1, 64), _log(rng, 1024, 16384),
                     _log(rng, 1024, 16384, 16))
    if family == "tokens":
        return _gemm("", rng.choice(["i8", "f16"]), _log(rng, 65, 512), _log(rng, 1024, 12288), _log(rng, 1024, 12288, 64))
    if family == "large":
        return _gemm("", rng.choice(["i8", "f16", "bf16"]), _log(rng, 512, 8192), _log(rng, 512, 12288),
                     _log(rng, 512, 12288, 16))
    if family == "layout":    # K-major operands
        return _gemm("", rng.choice(["i8", "f16", "bf16"]), _log(rng, 256, 8192, 16), _log(rng, 256, 8192, 16),
                     _log(rng, 256, 8192, 16), rng.choice(["mk_kn", "mk_kn", "km_nk", "km_kn"]))
    if family == "ragged":    # no extent a whole 16-byte vector
        return _gemm("", rng.choice(["i8", "f16", "f16", "bf16"]), _log(rng, 32, 4096), _log(rng, 32, 4096) | 1,
                     _log(rng, 64, 4096) | 1, rng.choice(["mk_nk", "mk_nk", "mk_kn", "km_nk"]))
    if family == "conv":
        f = rng.choice([1, 1, 3, 3, 5])
        dtype = rng.choice(["i8", "f16"])
        return _conv("", dtype, _log(rng, 1, 256), _log(rng, 16, 1024, 16), _log(rng, 16, 1024, 8), _log(rng, 7, 112), f,
                     rng.choice([1, 1, 2]), f // 2, fused=rng.choice(["", "bias_relu", "bias_relu_add"]) if dtype == "f16" else "")
    if family == "odd_conv":  # first layers: 1 ... 6 channels (RGB, RGB + depth, grey)
        f = rng.choice([3, 3, 5, 7])
        dtype = rng.choice(["i8", "f16"])
        return _conv("", dtype, _log(rng, 1, 128), rng.choice([1, 3, 3, 3, 4, 5, 6]), _log(rng, 16, 96, 8),
                     _log(rng, 28, 256), f, rng.choice([1, 2, 2]), f // 2, fused=rng.choice(["", "bias_relu"]) if dtype == "f16" else "")
    if family == "conv3d":
        return _conv("", rng.choice(["i8", "f16", "f16"]), _log(rng, 1, 32), _log(rng, 16, 256, 16), _log(rng, 16, 256, 16),
                     _log(rng, 8, 48), 3, rng.choice([1, 1, 2]), 1, ndim=3)
    if family == "gemm_gemm":
        d = rng.choice([32, 64, 64, 128])
        return _gemm_gemm("", _log(rng, 8, 256), _log(rng, 64, 2048), _log(rng, 64, 2048), d, d)
    d = rng.choice([32, 64, 64, 80, 128, 128])
    m = _log(rng, 128, 4096)
    mask = rng.random() < 0.5
    return _gemm_gemm("", _log(rng, 8, 256), m, m if mask or rng.random() < 0.5 else _log(rng, 128, 4096), d, d, True, mask)


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    least = min(_cost(c) for c in listed()) / 16
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw_one(rng)
        if least <= _cost(c) <= most and max(_operand_bytes(c)) < (1 << 31) - (1 << 20):
            del c["name"]
            return c


# ------------------------------------------------------------------------------------------------ sizes
def _es(case):
    return 1 if case["dtype"] == "i8" else 2


def _out_hw(case):
    return (case["hw"] + 2 * case["pad"] - ((case["f"] - 1) * case["dil"] + 1)) // case["stride"] + 1


def _elements(case):
    """(elements of every input, elements of the output) that a pass has to touch."""
    if case["kind"] == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return [M * K, N * K], M * N
    if case["kind"] == "conv":
        nd, ho = case["ndim"], _out_hw(case)
        side = ho if case["f"] == 1 else case["hw"]  # (a strided 1x1 filter reads the pixels it lands on)
        out = case["N"] * ho ** nd * case["K"]
        ins = [case["N"] * side ** nd * case["C"], case["K"] * case["f"] ** nd * case["C"]]
        return ins + [case["K"]] * (case["fused"] != "") + [out] * (case["fused"] == "bias_relu_add"), out
    G, M, N, K, O = (case[k] for k in "GMNKO")
    return [G * M * K, G * N * K, G * N * O], G * M * O


def _operand_bytes(case):
    ins, out = _elements(case)
    return [x * _es(case) for x in ins + [out]] + \
        ([case["N"] * case["hw"] ** case["ndim"] * case["C"] * _es(case)] if case["kind"] == "conv" else [])


def work(case):
    ins, out = _elements(case)
    if case["kind"] == "gemm":
        flops = 2.0 * case["M"] * case["N"] * case["K"]
    elif case["kind"] == "conv":
        flops = 2.0 * out * case["C"] * case["f"] ** case["ndim"]
    else:
        M, N = case["M"], case["N"]
        scores = sum(min(m + 1, N) for m in range(M)) if case["mask"] else M * N
        flops = 2.0 * case["G"] * scores * (case["K"] + case["O"])
    return {"bytes": float((sum(ins) + out) * _es(case)), "flops": flops}


def tolerance(case):
    """Integers come back bit for bit. 16-bit results are fp32 sums rounded once: against the same problem in 64 bits the
    fp16 GEMM and conv outputs differ by 2.1e-4 (2-norm), bf16 by 1.7e-3, the fused pair (whose intermediate is rounded
    to fp16 as well) by 2.9e-4 and attention by 2.6e-4 ... 2.8e-4; the largest single difference is half a unit of the last
    place (4.9e-4 / 3.9e-3), up to 2.9e-3 where an intermediate is rounded first. About four times that is stated."""
    if case["dtype"] == "i8":
        return "exact"
    if case["dtype"] == "bf16":
        return {"rel": 7e-3, "max": 1.6e-2}
    if case["kind"] == "gemm_gemm":
        return {"rel": 1.2e-3, "max": 1e-2}
    return {"rel": 8e-4, "max": 2e-3}


# ------------------------------------------------------------------------------------------------ one pass
def _normal(g, shape, dtype, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(scale).to(dtype)


def _quantised(g, shape):
    """int8 activations or weights as a symmetric quantiser leaves them: a quarter of the range per standard deviation."""
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(32.0).round_().clamp_(-127, 127).to(torch.int8)


def _requant(k):
    # accumulators of k products of the values above spread over about half of the int8 range
    return ck.RequantReluRequant(48.0 / (1024.0 * math.sqrt(k)), 0.7, rounded=True)


def _prepare_gemm(case, g):
    M, N, K = case["M"], case["N"], case["K"]
    la, lb = case["layout"].split("_")
    a_shape, b_shape = ((M, K) if la == "mk" else (K, M)), ((N, K) if lb == "nk" else (K, N))
    lay = dict(ALayout=ck.RowMajor if la == "mk" else ck.ColumnMajor, BLayout=ck.ColumnMajor if lb == "nk" else ck.RowMajor)
    if case["dtype"] == "i8":
        a, b, op, cop = _quantised(g, a_shape), _quantised(g, b_shape), ck.DeviceGemmInt8(**lay), _requant(K)
        c = torch.empty((M, N), device="cuda", dtype=torch.int8)
    else:
        dt = torch.float16 if case["dtype"] == "f16" else torch.bfloat16
        a, b, cop = _normal(g, a_shape, dt), _normal(g, b_shape, dt, K ** -0.5), ck.PassThrough()
        op = (ck.DeviceGemmF16 if case["dtype"] == "f16" else ck.DeviceGemmBF16)(**lay)
        c = torch.empty((M, N), device="cuda", dtype=dt)
    arg = op.MakeArgumentPointer(a, b, c, M, N, K, a_shape[1], b_shape[1], N, ck.PassThrough(), ck.PassThrough(), cop)
    return op, arg, c, (a, b)


def _prepare_conv(case, g):
    N, C, K, hw, f, nd = (case[k] for k in ("N", "C", "K", "hw", "f", "ndim"))
    ho = _out_hw(case)
    in_shape, wei_shape, out_shape = (N, *[hw] * nd, C), (K, *[f] * nd, C), (N, *[ho] * nd, K)
    geom = (N, K, C, [hw] * nd, [f] * nd, [ho] * nd, [case["stride"]] * nd, [case["dil"]] * nd, [case["pad"]] * nd,
            [case["pad"]] * nd)
    k = C * f ** nd
    if case["dtype"] == "i8":
        x, w = _quantised(g, in_shape), _quantised(g, wei_shape)
        y = torch.empty(out_shape, device="cuda", dtype=torch.int8)
        op = ck.DeviceConv2dFwdInt8() if nd == 2 else ck.DeviceConvNdFwdInt8(nd)
        return op, op.MakeArgumentPointer(x, w, y, *geom, ck.PassThrough(), ck.PassThrough(), _requant(k)), y, (x, w)
    x, w = _normal(g, in_shape, torch.float16), _normal(g, wei_shape, torch.float16, k ** -0.5)
    y = torch.empty(out_shape, device="cuda", dtype=torch.float16)
    if not case["fused"]:
        op = ck.DeviceConv2dFwdF16() if nd == 2 else ck.DeviceConvNdFwdF16(nd)
        return op, op.MakeArgumentPointer(x, w, y, *geom, ck.PassThrough(), ck.PassThrough(), ck.PassThrough()), y, (x, w)
    op, bias = ck.DeviceConv2dFwdBiasActivationF16(), _normal(g, (K,), torch.float16)
    if case["fused"] == "bias_relu":
        return op, op.MakeArgumentPointer(x, w, y, bias, *geom, ck.PassThrough(), ck.PassThrough(), ck.AddRelu()), y, (x, w, bias)
    r = _normal(g, out_shape, torch.float16)
    return op, op.MakeArgumentPointer(x, w, y, bias, r, *geom, ck.PassThrough(), ck.PassThrough(), ck.AddReluAdd()), y, (x, w, bias, r)


def _prepare_gemm_gemm(case, g):
    G, M, N, K, O = (case[k] for k in "GMNKO")
    a, b1 = _normal(g, (G, M, K), torch.float16), _normal(g, (G, N, O), torch.float16, 1.0 if case["softmax"] else N ** -0.5)
    b0 = _normal(g, (G, N, K), torch.float16, 1.0 if case["softmax"] else K ** -0.5)
    c = torch.empty((G, M, O), device="cuda", dtype=torch.float16)
    dims = (M, N, K, O, G, K, K, O, O, M * K, N * K, N * O, M * O)
    if case["softmax"]:
        op = ck.DeviceBatchedGemmSoftmaxGemmF16(MaskOutUpperTriangle=case["mask"])
        arg = op.MakeArgumentPointer(a, b0, b1, c, *dims, ck.PassThrough(), ck.PassThrough(), ck.Scale(K ** -0.5))
    else:
        op = ck.DeviceBatchedGemmGemmF16()
        arg = op.MakeArgumentPointer(a, b0, b1, c, *dims)
    return op, arg, c, (a, b0, b1)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    make = {"gemm": _prepare_gemm, "conv": _prepare_conv, "gemm_gemm": _prepare_gemm_gemm}[case["kind"]]
    op, arg, out, operands = make(case, g)
    if not op.IsSupportedArgument(arg):
        raise ValueError(op.GetTypeString() + ": " + ck.capi.last_error())
    need = op.GetWorkSpaceSize(arg)
    if need:
        op.SetWorkSpacePointer(arg, torch.empty(need, device="cuda", dtype=torch.uint8))
    return {"invoker": op.MakeInvokerPointer(), "argument": arg, "out": out, "operands": operands,
            "config": ck.StreamConfig(torch.cuda.current_stream().cuda_stream)}


def run(state):
    state["invoker"].Run(state["argument"], state["config"])
    return state["out"]
