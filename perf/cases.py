"""The work a user of this framework has it do, as timed cases.

Seven kinds of pass, each through the public entry points (`amdmigraphx_amd.ops`, or a program of
`amdmigraphx_amd.migraphx` compiled for the target):

  linear     a quantized linear layer, activations in and activations out: quantizelinear of the float input,
             quant_dot with the dequantizing epilogue and the bias (int8 or fp8; decode rows over weights
             reordered ahead of time, prefill rows over the [K, N] or [N, K] matrix)
  w4         an int4 weight-only linear layer on half activations
  attention  the two batched products of an attention layer whose dots were quantized
  conv       a quantized convolution with the dequantizing epilogue
  mx         a product of block-scaled (fp4 or fp8) operands
  codec      tensors stored quantized and read back: quantize -> dequantize, or 4-bit packed
  encoder    a compiled int8 QDQ encoder program: gather, layer norms, attention, GELU and all

Sizes are those of the benchmark's configurations (hidden 768 / 4096 / 8192, feed-forward 3072 / 14336 /
28672, vocabulary 30522, 32 x 384 tokens) and log-uniform ranges around them."""
import math

import numpy as np
import torch

from amdmigraphx_amd import migraphx as mgx
from amdmigraphx_amd import ops
from amdmigraphx_amd.capi import DT, lib

_FLOAT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2, "int8": 1, "fp8": 1}


def _linear(m, k, n, dtype, out, weights="nk", scale="tensor", zero_point=False):
    """weights: "nk" as a torch linear layer stores them, "kn" as an ONNX MatMul does; scale: of the
    activations, one for the tensor or one per row (token); zero_point: asymmetric int8 activations."""
    return {"kind": "linear", "m": m, "k": k, "n": n, "dtype": dtype, "out": out, "weights": weights,
            "scale": scale, "zero_point": zero_point}


def _w4(m, k, n, group=128, zero_points=False):
    return {"kind": "w4", "m": m, "k": k, "n": n, "group": group, "zero_points": zero_points}


def _attention(batch, seq, head, dtype, out):
    return {"kind": "attention", "batch": batch, "seq": seq, "head": head, "dtype": dtype, "out": out}


def _conv(n, c, hw, o, window, stride, group, dtype, out):
    return {"kind": "conv", "n": n, "c": c, "hw": hw, "o": o, "window": window, "stride": stride, "group": group,
            "dtype": dtype, "out": out}


def _mx(m, k, n, dtype):
    return {"kind": "mx", "m": m, "k": k, "n": n, "dtype": dtype}


def _codec(rows, cols, dtype, code, scale):
    return {"kind": "codec", "rows": rows, "cols": cols, "dtype": dtype, "code": code, "scale": scale}


def _encoder(batch, seq, hidden):
    return {"kind": "encoder", "batch": batch, "seq": seq, "hidden": hidden, "layers": 2}


def listed():
    return [
        # one token of a decode loop through a square projection: the smallest call, launch and host latency
        dict(_linear(1, 4096, 4096, "int8", "bf16"), name="linear_int8_m1"),
        # a batch of one sequence onto a vocabulary: a width no tile divides, weights as ONNX stores them,
        # activations with a zero point
        dict(_linear(500, 768, 30522, "int8", "f32", "kn", zero_point=True), name="linear_int8_vocab"),
        # a chunk of a prompt, or many sequences decoded together: too few rows to fill the chip
        dict(_linear(128, 8192, 8192, "fp8", "bf16", "kn"), name="linear_fp8_m128"),
        # a long prompt through the widest projection, one scale per token: the largest
        dict(_linear(2048, 8192, 28672, "fp8", "bf16", "kn", "row"), name="linear_fp8_m2048"),
        # decode of one sequence: streams the packed weights
        dict(_w4(1, 4096, 14336), name="w4_m1"),
        # decode of a batch of sequences
        dict(_w4(48, 14336, 4096), name="w4_m48"),
        # prefill
        dict(_w4(2048, 4096, 14336), name="w4_m2048"),
        # 8 images of 197 patches in 12 heads: rows of 197 bytes, aligned to nothing
        dict(_attention(96, 197, 64, "int8", "f32"), name="attention_int8_s197"),
        # an image network's early 3 x 3 layer
        dict(_conv(32, 64, 56, 64, 3, 1, 1, "int8", "f32"), name="conv3x3_int8"),
        # block-scaled weights and activations
        dict(_mx(512, 4096, 4096, "fp4"), name="mx_fp4_m512"),
        # a cache of keys and values stored in 4 bits and read back
        dict(_codec(8192, 1024, "bf16", "int4", "row"), name="codec_int4"),
        # the encoder of the benchmark at its full batch, two of its layers
        dict(_encoder(32, 384, 768), name="encoder_b32_s384"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _to(v, step):
    return max(step, v // step * step)


def _kind(rng):
    """Kinds in the proportion of the listed cases."""
    return rng.choice(["linear"] * 4 + ["w4"] * 3 + ["attention", "conv", "mx", "codec", "encoder"])


def draw(rng):
    """One more case: sizes over the logarithm of their range, a good part of them odd; never more work than
    the largest listed case (or the listed encoder, for an encoder)."""
    kind = _kind(rng)
    while True:
        case = _draw(rng, kind)
        w = work(case)
        if w["flops"] <= 9.6e11 and w["bytes"] <= 3.8e8:
            return case


def _draw(rng, kind):
    if kind == "linear":
        m = _log(rng, 1, 8192)
        k = _to(_log(rng, 256, 14336), rng.choice([512, 512, 64, 64, 8, 1]))
        n = _to(_log(rng, 256, 30522), rng.choice([512, 512, 64, 64, 4, 1]))
        dtype = rng.choice(["int8", "fp8"])
        scale = rng.choice(["tensor", "tensor", "row"])
        zero_point = dtype == "int8" and scale == "tensor" and rng.random() < 0.25
        return _linear(m + (m == k), k, n, dtype, rng.choice(["bf16", "bf16", "f16", "f32"]),
                       rng.choice(["nk", "kn"]), scale, zero_point)
    if kind == "w4":
        group = rng.choice([128, 128, 128, 64, 32])
        m = _log(rng, 1, 4096)
        # group sizes below 128 and zero points per group are those of smaller layers
        small = group < 128
        k = _to(_log(rng, 512, 4096 if small else 14336), rng.choice([512, 512, 128]))
        n = _to(_log(rng, 512, 4096 if small else 28672), rng.choice([512, 128, 16]))
        return _w4(min(m, 256) if small else m, k, n, group, rng.random() < 0.25)
    if kind == "attention":
        return _attention(_log(rng, 8, 384), _log(rng, 16, 1024), rng.choice([32, 64, 64, 128]),
                          rng.choice(["int8", "int8", "fp8"]), rng.choice(["f32", "f16", "bf16"]))
    if kind == "conv":
        hw = _log(rng, 7, 128)
        c = _to(_log(rng, 8, 1024), rng.choice([64, 64, 16, 8]))
        depthwise = rng.random() < 0.2
        o = c if depthwise else _to(_log(rng, 16, 1024), rng.choice([64, 16]))
        window = rng.choice([3, 5]) if depthwise else rng.choice([1, 3, 3, 5])
        return _conv(_log(rng, 1, 64), c, hw, o, window, rng.choice([1, 1, 2]), c if depthwise else 1,
                     "int8" if depthwise else rng.choice(["int8", "int8", "fp8"]), rng.choice(["f32", "f32", "f16"]))
    if kind == "mx":
        return _mx(_log(rng, 16, 4096), _to(_log(rng, 512, 14336), 128), _to(_log(rng, 512, 14336), 64),
                   rng.choice(["fp4", "fp8"]))
    if kind == "codec":
        code = rng.choice(["int8", "fp8", "int4"])
        cols = _log(rng, 64, 8192)
        rows = _log(rng, 16, 16384)
        return _codec(rows + (rows == cols), cols // 2 * 2 if code == "int4" else cols,
                      rng.choice(["bf16", "f16", "f32"]), code, rng.choice(["tensor", "row", "col"]))
    return _encoder(_log(rng, 1, 32), _log(rng, 16, 384), rng.choice([256, 512, 768]))


# ---- inputs ----------------------------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _codes(x, dtype, scale):
    """int8 codes, or fp8 e4m3fn codes as bytes, of x / scale."""
    if dtype == "int8":
        return (x / scale).round_().clamp_(-127, 127).to(torch.int8)
    return (x / scale).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)


def _top(dtype):
    return 127.0 if dtype == "int8" else 448.0


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, _generator(seed))


def _prepare_linear(case, g):
    m, k, n, dtype = case["m"], case["k"], case["n"], case["dtype"]
    out = _FLOAT[case["out"]]
    # activations in the layer's own float type (a float32 graph, or a 16-bit one)
    x = _normal(g, m, k).to(out)
    w = _normal(g, n, k, std=0.02)
    sw = w.abs().amax(1) / _top(dtype)
    w = _codes(w, dtype, sw[:, None])
    if case["weights"] == "kn":
        w = w.t().contiguous().t()
    fp8 = dtype == "fp8"
    zp = 0
    if case["scale"] == "row":
        sx = x.float().abs().amax(1) / _top(dtype)
    elif case["zero_point"]:
        lo, hi = x.float().amin(), x.float().amax()
        sx = ((hi - lo) / 255.0).reshape(1)
        zp = -7
    else:
        sx = (x.float().abs().amax() / _top(dtype)).reshape(1)
    sx = sx.to(out)
    bt = w.t()  # [K, N]: a view of either storage
    s = {"case": case, "x": x, "sx": sx, "sx32": sx.float(), "w": bt, "sw": sw.contiguous(),
         "bias": _normal(g, n, std=0.02), "zp": zp, "out": out,
         "zp_tensor": torch.tensor([zp], dtype=torch.int8, device="cuda") if zp else None,
         "colsum": ops.colsum_i8(bt) if zp else None}
    # constant weights are reordered once where few rows will meet them, as the target does on compile
    s["packed"] = ops.quant_dot_prepack(bt, fp8) if m <= 16 else None
    need = 0 if s["packed"] is not None else ops.quant_dot_workspace_size(m, n, k, trans_b=case["weights"] == "nk",
                                                                          fp8=fp8)
    s["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    return s


def _prepare_w4(case, g):
    m, k, n, group = case["m"], case["k"], case["n"], case["group"]
    w = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8, device="cuda")
    scales = (torch.rand(n, k // group, generator=g, device="cuda") * 0.015 + 0.005).half()
    zp = torch.randint(0, 16, (n, k // group), generator=g, dtype=torch.uint8, device="cuda") \
        if case["zero_points"] else 8
    s = {"case": case, "x": _normal(g, m, k).half(), "w": w, "scales": scales, "zp": zp, "packed": None,
         "workspace": None}
    if not case["zero_points"] and lib().mi355_w4a16_prepacked_max_rows(n, k, group) >= m:
        s["packed"] = ops.w4a16_prepack(w, scales, group, 8)
    if s["packed"] is None:
        need = ops.w4a16_gemm_workspace_size(m, n, k, group)
        s["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    return s


def _prepare_attention(case, g):
    b, s, d, dtype = case["batch"], case["seq"], case["head"], case["dtype"]
    q, k, v = (_normal(g, b, s, d) for _ in range(3))
    p = torch.softmax(torch.bmm(q, k.transpose(1, 2).contiguous()) / math.sqrt(d), dim=2)
    scales = [(t.abs().amax() / _top(dtype)).reshape(1) for t in (q, k, p, v)]
    return {"case": case, "codes": [_codes(t, dtype, sc) for t, sc in zip((q, k, p, v), scales)], "scales": scales}


def _prepare_conv(case, g):
    n, c, hw, o, kw, group, dtype = (case[x] for x in ("n", "c", "hw", "o", "window", "group", "dtype"))
    x = _normal(g, n, c, hw, hw).clamp_(min=0)  # behind a ReLU
    w = _normal(g, o, c // group, kw, kw, std=0.05)
    sx = (x.amax() / _top(dtype)).reshape(1)
    sw = (w.abs().amax((1, 2, 3)) / _top(dtype)).contiguous()
    return {"case": case, "x": _codes(x, dtype, sx), "w": _codes(w, dtype, sw[:, None, None, None]), "sx": sx, "sw": sw}


def _prepare_mx(case, g):
    m, k, n, fp4 = case["m"], case["k"], case["n"], case["dtype"] == "fp4"

    def codes(rows):
        if fp4:
            return torch.randint(0, 256, (rows, k // 2), generator=g, dtype=torch.uint8, device="cuda")
        return _normal(g, rows, k, std=64.0).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)

    def scales(rows):
        return torch.exp2(torch.randint(-9, -4, (rows, k // 32), generator=g, device="cuda").float())

    return {"case": case, "a": codes(m), "b": codes(n), "sa": scales(m), "sb": scales(n)}


def _prepare_codec(case, g):
    rows, cols = case["rows"], case["cols"]
    x = _normal(g, rows, cols).to(_FLOAT[case["dtype"]])
    top = {"int8": 127.0, "fp8": 448.0, "int4": 7.0}[case["code"]]
    a = x.float().abs()
    a = {"tensor": lambda: a.amax().reshape(1), "row": lambda: a.amax(1), "col": lambda: a.amax(0)}[case["scale"]]()
    s = {"case": case, "x": x, "scale": (a / top).to(x.dtype), "zp": None}
    if case["code"] == "int4":
        s["zp"] = torch.full_like(a, 8).to(torch.uint8)
    return s


def _encoder_weights(case, g):
    """Float weights as int8 codes with a scale per column, biases, and the token ids."""
    batch, seq, hidden, vocab = case["batch"], case["seq"], case["hidden"], 30522

    def linear(n_in, n_out):
        w = _normal(g, n_in, n_out, std=0.02)
        sw = w.abs().amax(0) / 127.0
        return _codes(w, "int8", sw), sw, _normal(g, n_out, std=0.02)

    def norm():
        return torch.rand(hidden, generator=g, device="cuda") * 0.2 + 0.9, _normal(g, hidden, std=0.02)

    return {"words": _normal(g, vocab, hidden, std=0.02), "positions": _normal(g, seq, hidden, std=0.02),
            "norm": norm(),
            "layers": [{"q": linear(hidden, hidden), "k": linear(hidden, hidden), "v": linear(hidden, hidden),
                        "o": linear(hidden, hidden), "norm1": norm(), "up": linear(hidden, 4 * hidden),
                        "down": linear(4 * hidden, hidden), "norm2": norm()} for _ in range(case["layers"])],
            "ids": torch.randint(0, vocab, (batch * seq,), generator=g, dtype=torch.int32, device="cuda")}


# largest activation in front of each of an encoder layer's linears, as calibration leaves them
_AMAX = {"x": 4.5, "context": 0.5, "up": 2.5}


def _prepare_encoder(case, g):
    batch, seq, hidden, heads, ffn, d = (case["batch"], case["seq"], case["hidden"], case["hidden"] // 64,
                                         case["hidden"] * 4, 64)
    tokens = batch * seq
    weights = _encoder_weights(case, g)
    p = mgx.program()
    mm = p.get_main_module()

    def host(t):
        return np.ascontiguousarray(t.cpu().numpy())

    def op(name, *args, **attributes):
        return mm.add_instruction(mgx.op(name, **attributes), list(args))

    def lit(v):
        return mm.add_literal(v)

    def over(v, lens):
        return op("multibroadcast", v, out_lens=lens)

    def row(v, lens):
        return op("broadcast", v, axis=1, out_lens=lens)

    def scalar(v, lens):
        return over(lit(np.float32([v])), lens)

    def layer_norm(x, norm):
        lens = [tokens, hidden]
        mean = over(op("reduce_mean", x, axes=[-1]), lens)
        xc = op("sub", x, mean)
        var = op("reduce_mean", op("mul", xc, xc), axes=[-1])
        rs = op("rsqrt", op("add", var, scalar(1e-5, [tokens, 1])))
        y = op("mul", xc, over(rs, lens))
        return op("add", op("mul", y, row(lit(host(norm[0])), lens)), row(lit(host(norm[1])), lens))

    def quantized(x, width, amax):
        s, z = lit(np.float32([amax / 127.0])), lit(np.int8([0]))
        lens = [tokens, width]
        q = op("quantizelinear", x, over(s, lens), over(z, lens))
        return op("dequantizelinear", q, over(s, lens), over(z, lens))

    def linear(x, wsb):
        w, sw, bias = wsb
        lens = list(w.shape)
        w = op("dequantizelinear", lit(host(w)), row(lit(host(sw)), lens), row(lit(np.zeros(lens[1], np.int8)), lens))
        return op("add", op("dot", x, w), row(lit(host(bias)), [tokens, lens[1]]))

    def split(x):
        x = op("reshape", x, dims=[batch, seq, heads, d])
        return op("contiguous", op("transpose", x, permutation=[0, 2, 1, 3]))

    def gelu(x, lens):
        e = op("erf", op("mul", x, scalar(math.sqrt(0.5), lens)))
        return op("mul", op("mul", x, scalar(0.5, lens)), op("add", e, scalar(1.0, lens)))

    def layer(x, w):
        lens = [tokens, hidden]
        xin = quantized(x, hidden, _AMAX["x"])
        q, k, v = (split(linear(xin, w[name])) for name in "qkv")
        scores = op("dot", q, op("transpose", k, permutation=[0, 1, 3, 2]))
        scores = op("mul", scores, scalar(1.0 / math.sqrt(d), [batch, heads, seq, seq]))
        ctx = op("dot", op("softmax", scores, axis=3), v)
        ctx = op("contiguous", op("transpose", ctx, permutation=[0, 2, 1, 3]))
        att = linear(quantized(op("reshape", ctx, dims=lens), hidden, _AMAX["context"]), w["o"])
        x = layer_norm(op("add", x, att), w["norm1"])
        h = gelu(linear(quantized(x, hidden, _AMAX["x"]), w["up"]), [tokens, ffn])
        return layer_norm(op("add", x, linear(quantized(h, ffn, _AMAX["up"]), w["down"])), w["norm2"])

    ids = mm.add_parameter("ids", mgx.shape(type="int32_type", lens=[tokens]))
    x = op("gather", lit(host(weights["words"])), ids, axis=0)
    pos = over(lit(host(weights["positions"])), [batch, seq, hidden])
    x = op("reshape", op("add", op("reshape", x, dims=[batch, seq, hidden]), pos), dims=[tokens, hidden])
    x = layer_norm(x, weights["norm"])
    for w in weights["layers"]:
        x = layer(x, w)
    mm.add_return([x])
    p.compile(mgx.get_target("gpu"), offload_copy=False)
    return {"case": case, "program": p, "parameters": {"ids": mgx.to_gpu(mgx.argument(host(weights["ids"])))}}


_PREPARE = {"linear": _prepare_linear, "w4": _prepare_w4, "attention": _prepare_attention, "conv": _prepare_conv,
            "mx": _prepare_mx, "codec": _prepare_codec, "encoder": _prepare_encoder}


# ---- one pass --------------------------------------------------------------------------------------------


def run(s):
    return _RUN[s["case"]["kind"]](s, s["case"])


def _run_linear(s, case):
    fp8 = case["dtype"] == "fp8"
    q = ops.quantizelinear(s["x"], s["sx"], s["zp_tensor"], DT.FP8 if fp8 else DT.I8)
    args = dict(fp8=fp8, scale_a=s["sx32"], scale_b=s["sw"], zp_a=s["zp"], colsum_b=s["colsum"], out_dtype=s["out"],
                bias=s["bias"])
    if s["packed"] is not None:
        return ops.quant_dot_prepacked(q, s["packed"], case["n"], **args)
    return ops.quant_dot(q, s["w"], workspace=s["workspace"], **args)


def _run_w4(s, case):
    if s["packed"] is not None:
        return ops.w4a16_gemm_prepacked(s["x"], s["packed"], case["n"])
    return ops.w4a16_gemm(s["x"], s["w"], s["scales"], case["group"], s["zp"], workspace=s["workspace"])


def _run_attention(s, case):
    q, k, p, v = s["codes"]
    sq, sk, sp, sv = s["scales"]
    args = dict(fp8=case["dtype"] == "fp8", out_dtype=_FLOAT[case["out"]])
    return {"scores": ops.quant_dot(q, k.transpose(1, 2), scale_a=sq, scale_b=sk, **args),
            "context": ops.quant_dot(p, v, scale_a=sp, scale_b=sv, **args)}


def _run_conv(s, case):
    pad = case["window"] // 2
    return ops.quant_convolution(s["x"], s["w"], padding=(pad, pad), stride=(case["stride"],) * 2, group=case["group"],
                                 fp8=case["dtype"] == "fp8", scale_x=s["sx"], scale_w=s["sw"],
                                 out_dtype=_FLOAT[case["out"]])


def _run_mx(s, case):
    fp4 = case["dtype"] == "fp4"
    return ops.quant_dot_mx(s["a"], s["b"], s["sa"], s["sb"], a_fp4=fp4, b_fp4=fp4)


def _run_codec(s, case):
    code = {"int8": DT.I8, "fp8": DT.FP8, "int4": DT.U8}[case["code"]]
    stored = ops.quantizelinear(s["x"], s["scale"], s["zp"], code)
    if case["code"] != "int4":
        return {"stored": stored, "read": ops.dequantizelinear(stored, s["scale"], x_type=code)}
    stored = ops.pack_int4(stored)
    return {"stored": stored, "read": ops.dequantizelinear(ops.unpack_int4(stored), s["scale"], s["zp"])}


class _Device:
    """A program's result, which stays on the device, in the form torch takes without a copy."""

    def __init__(self, argument):
        shape = argument.get_shape()
        self.argument = argument
        self.__cuda_array_interface__ = {"shape": tuple(shape.lens()), "typestr": "<f4", "version": 2,
                                         "data": (argument.data_ptr(), False)}


def _run_encoder(s, case):
    return torch.as_tensor(_Device(s["program"].run(s["parameters"])[0]), device="cuda")


_RUN = {"linear": _run_linear, "w4": _run_w4, "attention": _run_attention, "conv": _run_conv, "mx": _run_mx,
        "codec": _run_codec, "encoder": _run_encoder}


# ---- the same in 64 bits ---------------------------------------------------------------------------------


def exact(case, seed):
    """What run() returns for these inputs, from plain torch in float64: the operands are the codes the operators
    are defined by (a quantized activation is rounded where its operator rounds it), all sums and scales double."""
    return _EXACT[case["kind"]](case, _generator(seed))


def _toward_zero(x, dtype):
    """float32 values cut to a 16-bit type's mantissa, as a quotient in that type is."""
    cut = {torch.float32: 0, torch.float16: 13, torch.bfloat16: 16}[dtype]
    return (x.view(torch.int32) >> cut << cut).view(torch.float32)


def _quantize(x, scale, code, zp=0):
    """quantizelinear's values (not their codes): of x's own type's quotient, and of a double one for fp8"""
    v = x.double() / scale.double()
    if code == "fp8":
        return v.clamp_(-448, 448).float().to(torch.float8_e4m3fn).double()
    lo, hi = {"int8": (-128, 127), "int4": (0, 15)}[code]
    return _toward_zero(v.float(), x.dtype).double().round_().add_(zp).clamp_(lo, hi)


def _values(codes, dtype):
    """int8 or fp8 codes as doubles"""
    return codes.double() if dtype == "int8" else codes.contiguous().view(torch.float8_e4m3fn).double()


def _exact_linear(case, g):
    s = _prepare_linear(case, g)
    sx = s["sx"][:, None] if case["scale"] == "row" else s["sx"]
    q = _quantize(s["x"], sx, case["dtype"], s["zp"]) - s["zp"]
    w = _values(s["w"].t(), case["dtype"])
    return torch.matmul(q, w.t()) * sx.double() * s["sw"].double() + s["bias"].double()


def _exact_w4(case, g):
    s = _prepare_w4(case, g)
    w = torch.stack([s["w"] & 15, s["w"] >> 4], dim=2).reshape(case["n"], -1, case["group"]).double()
    zp = s["zp"][:, :, None].double() if case["zero_points"] else 8
    w = (w - zp).mul_(s["scales"][:, :, None].double()).reshape(case["n"], case["k"])
    return torch.matmul(s["x"].double(), w.t())


def _exact_attention(case, g):
    s = _prepare_attention(case, g)
    q, k, p, v = (_values(c, case["dtype"]) * sc.double() for c, sc in zip(s["codes"], s["scales"]))
    return {"scores": torch.bmm(q, k.transpose(1, 2).contiguous()), "context": torch.bmm(p, v)}


def _exact_conv(case, g):
    s = _prepare_conv(case, g)
    pad, st, out = case["window"] // 2, case["stride"], (case["hw"] + 2 * (case["window"] // 2) - case["window"]) // \
        case["stride"] + 1
    x = torch.nn.functional.pad(_values(s["x"], case["dtype"]), (pad,) * 4)
    w = _values(s["w"], case["dtype"])
    total = 0
    for i in range(case["window"]):
        for j in range(case["window"]):
            tap = x[:, :, i:i + (out - 1) * st + 1:st, j:j + (out - 1) * st + 1:st]
            if case["group"] > 1:  # depthwise
                total = total + tap * w[:, 0, i, j][:, None, None]
            else:
                total = total + torch.matmul(w[:, :, i, j].contiguous(), tap.reshape(case["n"], case["c"], -1))
    return total.reshape(case["n"], case["o"], out, out) * (s["sx"].double() * s["sw"].double())[:, None, None]


def _exact_mx(case, g):
    s = _prepare_mx(case, g)
    fp4 = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device="cuda")
    fp4 = torch.cat([fp4, -fp4])

    def operand(codes, scales):
        if case["dtype"] == "fp4":
            v = fp4[torch.stack([codes & 15, codes >> 4], dim=2).long()].reshape(len(codes), -1)
        else:
            v = _values(codes, "fp8")
        return v * scales.double().repeat_interleave(32, dim=1)

    return torch.matmul(operand(s["a"], s["sa"]), operand(s["b"], s["sb"]).t())


def _exact_codec(case, g):
    s = _prepare_codec(case, g)
    scale = s["scale"][:, None] if case["scale"] == "row" else s["scale"]
    zp = 8 if case["code"] == "int4" else 0
    return {"stored": None, "read": (_quantize(s["x"], scale, case["code"], zp) - zp) * scale.double()}


def _exact_encoder(case, g):
    batch, seq, hidden, heads = case["batch"], case["seq"], case["hidden"], case["hidden"] // 64
    weights = _encoder_weights(case, g)

    def layer_norm(x, norm):
        x = x - x.mean(1, keepdim=True)
        x = x * torch.rsqrt((x * x).mean(1, keepdim=True) + float(np.float32(1e-5)))
        return x * norm[0].double() + norm[1].double()

    def linear(x, amax, wsb):
        scale = float(np.float32(amax / 127.0))
        w, sw, bias = (t.double() for t in wsb)
        return torch.matmul((x / scale).round().clamp(-128, 127), w) * (sw * scale) + bias

    def split(x):
        return x.reshape(batch, seq, heads, 64).transpose(1, 2).reshape(batch * heads, seq, 64)

    x = weights["words"].double()[weights["ids"].long()].reshape(batch, seq, hidden) + weights["positions"].double()
    x = layer_norm(x.reshape(batch * seq, hidden), weights["norm"])
    for w in weights["layers"]:
        q, k, v = (split(linear(x, _AMAX["x"], w[name])) for name in "qkv")
        p = torch.softmax(torch.bmm(q, k.transpose(1, 2).contiguous()) / 8.0, dim=2)
        context = torch.bmm(p, v).reshape(batch, heads, seq, 64).transpose(1, 2).reshape(batch * seq, hidden)
        x = layer_norm(x + linear(context, _AMAX["context"], w["o"]), w["norm1"])
        h = linear(x, _AMAX["x"], w["up"])
        h = h * 0.5 * (torch.erf(h * math.sqrt(0.5)) + 1.0)
        x = layer_norm(x + linear(h, _AMAX["up"], w["down"]), w["norm2"])
    return x


_EXACT = {"linear": _exact_linear, "w4": _exact_w4, "attention": _exact_attention, "conv": _exact_conv, "mx": _exact_mx,
          "codec": _exact_codec, "encoder": _exact_encoder}


# ---- what a pass cannot do without ---------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n, f = case["m"], case["k"], case["n"], _SIZE[case["out"]]
        return {"bytes": m * k * f + k * n + 8 * n + m * n * f, "flops": 2 * m * k * n}
    if kind == "w4":
        m, k, n = case["m"], case["k"], case["n"]
        per_group = 3 if case["zero_points"] else 2
        return {"bytes": 2 * m * k + k * n // 2 + per_group * n * (k // case["group"]) + 2 * m * n,
                "flops": 2 * m * k * n}
    if kind == "attention":
        b, s, d, f = case["batch"], case["seq"], case["head"], _SIZE[case["out"]]
        return {"bytes": b * (3 * s * d + s * s + f * (s * s + s * d)), "flops": 4 * b * s * s * d}
    if kind == "conv":
        n, c, hw, o, kw, group = (case[x] for x in ("n", "c", "hw", "o", "window", "group"))
        out = (hw + 2 * (kw // 2) - kw) // case["stride"] + 1
        taps = c // group * kw * kw
        return {"bytes": n * c * hw * hw + o * taps + 4 * o + n * o * out * out * _SIZE[case["out"]],
                "flops": 2 * n * o * out * out * taps}
    if kind == "mx":
        m, k, n = case["m"], case["k"], case["n"]
        per_row = (k // 2 if case["dtype"] == "fp4" else k) + k // 32 * 4
        return {"bytes": (m + n) * per_row + 4 * m * n, "flops": 2 * m * k * n}
    if kind == "codec":
        count, f = case["rows"] * case["cols"], _SIZE[case["dtype"]]
        # stored codes are written and read back
        stored = count // 2 if case["code"] == "int4" else count
        return {"bytes": 2 * count * f + 2 * stored, "flops": 4 * count}
    tokens, hidden, layers, seq = case["batch"] * case["seq"], case["hidden"], case["layers"], case["seq"]
    return {"bytes": tokens * 4 + 8 * tokens * hidden + layers * 12 * hidden * hidden,
            "flops": layers * (2 * tokens * 12 * hidden * hidden + 4 * tokens * seq * hidden)}


def tolerance(case):
    """int8 products and convolutions and the codecs are whole numbers, double products and roundings that are
    pinned down bit for bit.  The others sum in float32: about four times what a pass differs by from the same
    sums in float64 (a 16-bit result then also flips a last bit here and there, which is its largest error).
    Measured: fp8 1.5e-5 as float32, 8e-5 as half, 2.9e-4 as bfloat16; int4 weights 1.5e-5; mx 1.5e-5."""
    kind = case["kind"]
    if kind == "encoder":
        # a last bit carries an activation across a step of its int8 grid: attention summed in float32 in place
        # of float64 moves the result by 1.7e-3 and at most 3.2e-2
        return {"rel": 7e-3, "max": 0.13}
    if kind == "mx":
        return {"rel": 6e-5, "max": 1.2e-3}
    if kind == "w4":
        return {"rel": 6e-5, "max": 4e-3}
    if kind == "codec" or case["dtype"] == "int8":
        return "exact"
    return {"f32": {"rel": 6e-5, "max": 1.2e-3}, "f16": {"rel": 4e-4, "max": 4e-3},
            "bf16": {"rel": 1.2e-3, "max": 0.032}}[case["out"]]
