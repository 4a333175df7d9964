"""Performance cases of the quantized-inference path: what its users run, over the real ranges.

A case is a dict of plain values; `prepare` makes what a program holds before the call (inputs,
quantized weights, scales), `run` is one pass through the package's public entry points.  The
kinds of case:

  linear      a quantized linear on f32 activations, f32 result: quantize -> int8 GEMM ->
              dequantize, what replaces one nn.Linear of a model
  gemm        an int8 GEMM between two quantized operators (int8 in; int8, or f32 where an f32
              operator follows), dynamic number of rows
  weight_only floating-point activations times 8-bit weights: few rows when a model decodes,
              many when it reads its prompt
  bottleneck  a residual block of a quantized vision network: 1x1, 3x3 and 1x1 convolution,
              each with its activation fused, the block's input added at the end
  qdq         quantize and dequantize of an activation or a weight on their own
  calibrate   one observation step of post-training quantization: running min / max, scale and
              zero point, fake quantization
  encoder     a quantized BERT-base encoder layer, eager, as a service with dynamic sequence
              lengths runs it
"""
import math

import torch

from bladedisc_amd import bert_layer as B
from bladedisc_amd import kernels as K
from bladedisc_amd import observer as O

DEV = "cuda"

EPILOGUES = {"requant_cpu": K.EPI_REQUANT_CPU, "requant_gpu": K.EPI_REQUANT_GPU,
             "dequant_f32": K.EPI_DEQUANT_F32, "requant_dequant": K.EPI_REQUANT_CPU_DEQUANT_F32}
FLOATS = {"f32": torch.float32, "f16": torch.float16}
BYTES = {"f32": 4, "f16": 2, "int8": 1, "uint8": 1, "int16": 2}

# the most work a case may ask for: that of the largest listed one (4096^3)
MOST = 2.0 * 4096 ** 3 / 50


def listed():
    return [
        # one linear of a BERT-base layer on a short sequence: a launch or two, all latency
        dict(name="linear_64x768x768", kind="linear", m=64, k=768, n=768),
        # FFN2 of the same layer on a ragged batch of sequences
        dict(name="gemm_1000x3072x768", kind="gemm", m=1000, k=3072, n=768,
             epilogue="requant_cpu", bias=True, zx=0, dist="normal"),
        # no size a multiple of anything the tiles like, asymmetric activations, f32 result
        dict(name="gemm_odd_777x1000x1501", kind="gemm", m=777, k=1000, n=1501,
             epilogue="requant_dequant", bias=True, zx=-11, dist="normal"),
        # FFN1 at a large batch: wide result, short reduction
        dict(name="gemm_16384x768x3072", kind="gemm", m=16384, k=768, n=3072,
             epilogue="requant_cpu", bias=True, zx=0, dist="normal"),
        # the large square product: uniform operands, bias and requantisation fused
        dict(name="gemm_4096x4096x4096", kind="gemm", m=4096, k=4096, n=4096,
             epilogue="requant_gpu", bias=True, zx=0, dist="uniform"),
        # a decode step of sixteen sequences through a wide feed-forward projection
        dict(name="weight_only_16x4096x11008", kind="weight_only", m=16, k=4096, n=11008,
             dtype="f16", weight="uint8", bias=False),
        # a prompt through a square projection
        dict(name="weight_only_1024x4096x4096", kind="weight_only", m=1024, k=4096, n=4096,
             dtype="f16", weight="uint8", bias=True),
        # first stage of ResNet-50 at batch 32
        dict(name="bottleneck_32x56x64", kind="bottleneck", batch=32, size=56, channels=64),
        # a large activation, per tensor
        dict(name="qdq_16384x4096", kind="qdq", rows=16384, cols=4096, axis=-1, input="f32",
             dtype="int8"),
        # a small ragged one, asymmetric and per channel of the last axis
        dict(name="qdq_odd_1000x3073", kind="qdq", rows=1000, cols=3073, axis=1, input="f32",
             dtype="uint8"),
        # calibration on the activations of 8 sequences of 384 tokens
        dict(name="calibrate_3072x768", kind="calibrate", rows=3072, cols=768, axis=-1,
             symmetric=True),
        # an encoder layer at batch 8, sequence length 128, everything fused that can be
        dict(name="encoder_8x128", kind="encoder", batch=8, seq=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer's width: mostly a multiple of 64, now and then of 16, or anything."""
    v = _log(rng, lo, hi)
    step = rng.choice([64, 64, 64, 64, 16, 16, 1])
    return min(hi, max(lo, v - v % step))


def _draw(rng):
    kind = rng.choice(["linear", "gemm", "gemm", "gemm", "weight_only", "weight_only",
                       "bottleneck", "qdq", "qdq", "calibrate", "encoder"])
    if kind == "linear":
        return dict(kind=kind, m=_log(rng, 1, 4096), k=_width(rng, 256, 4096),
                    n=_width(rng, 256, 4096))
    if kind == "gemm":
        return dict(kind=kind, m=_log(rng, 1, 16384), k=_width(rng, 256, 4096),
                    n=_width(rng, 256, 4096), epilogue=rng.choice(sorted(EPILOGUES)),
                    bias=rng.random() < 0.7, zx=rng.choice([0, 0, 0, -11]),
                    dist=rng.choice(["normal", "normal", "uniform"]))
    if kind == "weight_only":
        return dict(kind=kind, m=_log(rng, 1, 2048), k=_width(rng, 512, 8192),
                    n=_width(rng, 512, 11008), dtype=rng.choice(["f16", "f16", "f16", "f32"]),
                    weight=rng.choice(["uint8", "uint8", "int8"]), bias=rng.random() < 0.5)
    if kind == "bottleneck":
        channels = rng.choice([64, 128, 256, 512])
        return dict(kind=kind, batch=_log(rng, 1, 32), channels=channels,
                    size=max(7, int(rng.uniform(0.7, 1.2) * 3584 / channels)))
    if kind == "qdq":
        dtype = rng.choice(["int8", "int8", "uint8", "int16"])
        return dict(kind=kind, rows=_log(rng, 16, 16384), cols=_width(rng, 64, 4096),
                    axis=rng.choice([-1, -1, 0, 1]), input=rng.choice(["f32", "f32", "f32", "f16"]),
                    dtype=dtype)
    if kind == "calibrate":
        return dict(kind=kind, rows=_log(rng, 64, 16384), cols=_width(rng, 64, 4096),
                    axis=rng.choice([-1, -1, 0]), symmetric=rng.random() < 0.7)
    return dict(kind=kind, batch=_log(rng, 1, 16), seq=_log(rng, 8, 384))


def draw(rng):
    """One more case of the kinds and ranges above, no larger than the largest listed one."""
    while True:
        case = _draw(rng)
        w = work(case)
        if max(w["bytes"], w["flops"] / 50) > MOST:
            continue
        if case["kind"] == "encoder" and case["batch"] * case["seq"] > 3072:
            continue
        return case


# ------------------------------------------------------------------------------- inputs
class _Maker:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device=DEV)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def ints(self, lo, hi, *shape, dtype=torch.int8):
        return torch.randint(lo, hi + 1, shape, generator=self.g, device=DEV, dtype=dtype)

    def normal_int8(self, std, *shape):
        """What a symmetric quantizer makes of a normal tensor."""
        return torch.clamp(torch.round(self.normal(*shape) * std), -127, 127).to(torch.int8)


def _f(v):
    return torch.tensor([float(v)], dtype=torch.float32, device=DEV)


def _i(v):
    return torch.tensor([int(v)], dtype=torch.int32, device=DEV)


def _prepare_linear(c, r):
    x = r.normal(c["m"], c["k"])
    w = r.normal(c["n"], c["k"]) * 0.02
    sx = x.abs().max().reshape(1) / 127
    sw = w.abs().amax(1) / 127
    w_q = K.quantize(w, sw, torch.zeros(c["n"], dtype=torch.int32, device=DEV), axis=0)
    so = _f(4.5 * 0.02 * math.sqrt(c["k"]) / 127)
    fused = c["m"] <= K.qlinear_f32_fused_max_rows(c["n"], c["k"])
    return dict(x=x, w=w_q, sx=sx, sw=sw, so=so, bias=r.normal(c["n"]) * 0.01, z=_i(0),
                fused=fused)


def _run_linear(s):
    if s["fused"]:
        return K.qlinear_f32(s["x"], s["w"], K.EPI_REQUANT_CPU_DEQUANT_F32, s["sx"], sw=s["sw"],
                             so=s["so"], bias=s["bias"])
    x_q = K.quantize(s["x"], s["sx"], s["z"])
    return K.qgemm(x_q, s["w"], K.EPI_REQUANT_CPU_DEQUANT_F32, sx=s["sx"], sw=s["sw"],
                   so=s["so"], bias=s["bias"])


def _prepare_gemm(c, r):
    m, k, n = c["m"], c["k"], c["n"]
    epi = EPILOGUES[c["epilogue"]]
    if c["dist"] == "uniform":
        a, w = r.ints(-127, 127, m, k), r.ints(-127, 127, n, k)
        sx, sw = _f(0.02), r.uniform(0.001, 0.05, n)
        lsb = 0.02 * 0.0255 * math.sqrt(k) * (127.0 * 128.0 / 3.0) / 40.0
    else:
        a, w = r.normal_int8(31.75, m, k), r.normal_int8(36.0, n, k)
        sx, sw = _f(1 / 31.75), r.uniform(0.9, 1.1, n) * (0.02 / 36.0)
        lsb = 4.5 * 0.02 * math.sqrt(k) / 127
    if c["zx"]:
        a = torch.clamp(a.to(torch.int16) + c["zx"], -128, 127).to(torch.int8)
    bias = None
    if c["bias"]:       # in units of the int8 output for requant_gpu, of the f32 result otherwise
        bias = r.normal(n) * 10.0 * (1.0 if c["epilogue"] == "requant_gpu" else lsb)
    return dict(a=a, w=w, epi=epi, sx=sx, sw=sw, bias=bias, zx=c["zx"],
                so=None if epi == K.EPI_DEQUANT_F32 else _f(lsb))


def _run_gemm(s):
    return K.qgemm(s["a"], s["w"], s["epi"], sx=s["sx"], sw=s["sw"], so=s["so"], bias=s["bias"],
                   zx=s["zx"])


def _prepare_weight_only(c, r):
    dt = FLOATS[c["dtype"]]
    signed = c["weight"] == "int8"
    w = r.normal(c["n"], c["k"]) * 30.0
    w = (torch.clamp(torch.round(w), -127, 127).to(torch.int8) if signed
         else torch.clamp(torch.round(w + 128.0), 0, 255).to(torch.uint8))
    zp = r.ints(-6, 6, c["n"], dtype=torch.int32) + (0 if signed else 128)
    return dict(x=r.normal(c["m"], c["k"]).to(dt), w=w, zp=zp,
                scale=(r.uniform(0.9, 1.1, c["n"]) * (0.02 / 30.0)).to(dt),
                bias=(r.normal(c["n"]) * 0.1).to(dt) if c["bias"] else None)


def _run_weight_only(s):
    return K.weight_only_qgemm(s["x"], s["w"], s["scale"], zero_points=s["zp"], bias=s["bias"])


def _relu_table(s_out):
    """int8 -> int8: dequantize, ReLU, quantize at the same scale."""
    z = _i(0)
    return K.activation_table(torch.relu, s_out, z, s_out, z)


def _prepare_bottleneck(c, r):
    nb, h, ch = c["batch"], c["size"], c["channels"]
    wide = 4 * ch
    md = list(K.NHWC_OHWI) + [1, 1, 1, 1, 1]
    # ReLU'd activations fill the non-negative half of the int8 range
    x = torch.clamp(torch.round(torch.relu(r.normal(nb, h, h, wide)) * 31.75), 0, 127).to(torch.int8)
    layers = []
    for ci, co, f in ((wide, ch, 1), (ch, ch, 3), (ch, wide, 1)):
        std = 1.0 / math.sqrt(0.5 * f * f * ci)              # keeps the activations at unit size
        layers.append(dict(w=r.normal_int8(36.0, co, f, f, ci),
                           sw=r.uniform(0.9, 1.1, co) * (std / 36.0), pad=[f // 2] * 4,
                           shape=[nb, h, h, co], bias=r.normal(co) * 0.05))
    s = _f(4.0 / 127)
    return dict(x=x, layers=layers, s=s, md=md, table=_relu_table(s), s_end=_f(6.0 / 127))


def _run_bottleneck(s):
    y = s["x"]
    one, two, three = s["layers"]
    table = K.make_postops(table=s["table"])
    for layer, post in ((one, table), (two, table),
                        (three, K.make_postops(residual=s["x"], residual_scale=s["s"], relu=True,
                                               out_scale=s["s_end"]))):
        y = K.qconv2d(y, layer["w"], layer["pad"], s["md"], layer["shape"], K.EPI_REQUANT_CPU,
                      sx=s["s"], sw=layer["sw"], so=s["s"], bias=layer["bias"], post=post)
    return y


def _prepare_qdq(c, r):
    rows, cols = c["rows"], c["cols"]
    x = (r.normal(rows, cols) * 2.0).to(FLOATS[c["input"]])
    axis = None if c["axis"] < 0 else c["axis"]
    n = 1 if axis is None else (rows, cols)[axis]
    qmin, qmax = {"int8": (-128, 127), "uint8": (0, 255), "int16": (-32768, 32767)}[c["dtype"]]
    scale = r.uniform(0.8, 1.2, n) * (16.0 / (qmax - qmin))
    zp = (torch.zeros(n, dtype=torch.int32, device=DEV) if c["dtype"] == "int16"
          else r.ints(-8, 8, n, dtype=torch.int32) + (qmin + qmax + 1) // 2)
    return dict(x=x, scale=scale, zp=zp, axis=axis, qmin=qmin, qmax=qmax,
                dtype=getattr(torch, c["dtype"]))


def _run_qdq(s):
    q = K.quantize(s["x"], s["scale"], s["zp"], axis=s["axis"], qmin=s["qmin"], qmax=s["qmax"],
                   dtype=s["dtype"])
    return q, K.dequantize(q, s["scale"], s["zp"], axis=s["axis"])


def _prepare_calibrate(c, r):
    per_channel = c["axis"] >= 0
    if per_channel:
        scheme = torch.per_channel_symmetric if c["symmetric"] else torch.per_channel_affine
    else:
        scheme = torch.per_tensor_symmetric if c["symmetric"] else torch.per_tensor_affine
    dtype = torch.qint8 if c["symmetric"] else torch.quint8
    ob = (O.PerChannelMinMaxObserver(c["axis"], dtype=dtype, qscheme=scheme) if per_channel
          else O.MinMaxObserver(dtype=dtype, qscheme=scheme))
    x = r.normal(c["rows"], c["cols"]) + (0.0 if c["symmetric"] else 0.5)
    return dict(ob=ob, x=x)


def _run_calibrate(s):
    y = s["ob"](s["x"])
    q = s["ob"].qparams
    return y, q.scale, q.zero_point, s["ob"].min_val, s["ob"].max_val


def _prepare_encoder(c, r, hidden=768, ffn=3072):
    g = lambda *shape: (r.normal(*shape) * 0.02).cpu().numpy()  # noqa: E731
    ones = torch.ones(hidden).numpy()
    zeros = torch.zeros(hidden).numpy()
    weights = dict(wq=g(hidden, hidden), wk=g(hidden, hidden), wv=g(hidden, hidden), bq=g(hidden),
                   bk=g(hidden), bv=g(hidden), wo=g(hidden, hidden), bo=g(hidden), ln1_g=ones,
                   ln1_b=zeros, w1=g(ffn, hidden), b1=g(ffn), w2=g(hidden, ffn), b2=g(hidden),
                   ln2_g=ones, ln2_b=zeros)
    layer = B.QuantBertLayer(weights, B.RawBackend(), fuse_epilogue=True)
    h = torch.nn.functional.layer_norm(r.normal(c["batch"], c["seq"], hidden), (hidden,))
    layer.calibrate(h)
    return dict(layer=layer, h=h)


def _run_encoder(s):
    return s["layer"].forward(s["h"])


_PREPARE = {"linear": _prepare_linear, "gemm": _prepare_gemm, "weight_only": _prepare_weight_only,
            "bottleneck": _prepare_bottleneck, "qdq": _prepare_qdq, "calibrate": _prepare_calibrate,
            "encoder": _prepare_encoder}
_RUN = {"linear": _run_linear, "gemm": _run_gemm, "weight_only": _run_weight_only,
        "bottleneck": _run_bottleneck, "qdq": _run_qdq, "calibrate": _run_calibrate,
        "encoder": _run_encoder}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, _Maker(seed))
    state["run"] = _RUN[case["kind"]]
    return state


def run(state):
    return state["run"](state)


def work(case):
    kind = case["kind"]
    if kind in ("linear", "gemm", "weight_only"):
        m, k, n = case["m"], case["k"], case["n"]
        if kind == "linear":
            size_in, size_out, per_n = 4, 4, 8
        elif kind == "gemm":
            size_in, per_n = 1, 4 + 4 * case["bias"]
            size_out = 1 if case["epilogue"] in ("requant_cpu", "requant_gpu") else 4
        else:
            size_in = size_out = BYTES[case["dtype"]]
            per_n = 4 + size_in * (1 + case["bias"])
        return dict(bytes=m * k * size_in + n * k + m * n * size_out + n * per_n,
                    flops=2 * m * k * n)
    if kind == "bottleneck":
        px, ch = case["batch"] * case["size"] ** 2, case["channels"]
        weights = 4 * ch * ch + 9 * ch * ch + 4 * ch * ch
        return dict(bytes=2 * px * 4 * ch + weights + 8 * 6 * ch, flops=2 * px * weights)
    if kind == "qdq":
        e = case["rows"] * case["cols"]
        n = 1 if case["axis"] < 0 else (case["rows"], case["cols"])[case["axis"]]
        return dict(bytes=e * (BYTES[case["input"]] + BYTES[case["dtype"]] + 4) + 8 * n, flops=4 * e)
    if kind == "calibrate":
        e = case["rows"] * case["cols"]
        return dict(bytes=8 * e, flops=6 * e)
    h, f, m = 768, 3072, case["batch"] * case["seq"]
    weights = 4 * h * h + 2 * h * f
    return dict(bytes=2 * 4 * m * h + weights + 8 * (4 * h + h + f + h),
                flops=2 * m * weights + 4 * m * case["seq"] * h)


def tolerance(case):
    kind = case["kind"]
    if kind == "weight_only":
        # one rounding to the result's type on top of an f32 accumulation
        return {"rel": 1e-3} if case["dtype"] == "f16" else {"rel": 1e-5}
    if kind == "gemm" and case["epilogue"] == "dequant_f32":
        return {"rel": 1e-6}
    if kind == "encoder":
        # the f32 attention and LayerNorm may round differently; an activation that lands on the
        # other side of a rounding tie then moves an int8 value, and with it a few outputs
        return {"rel": 2e-3, "max": 0.1}
    # integer sums and separately rounded f32 steps: every bit is defined
    return "exact"
