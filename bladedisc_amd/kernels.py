"""torch-tensor front-end of the raw kernel C ABI (include/disc_q8.h).

PyTorch only supplies device memory and the current stream here; every function
launches the hand-written HIP kernels in libdisc_q8_ral.so.  The operators go through
csrc_torch/torch_calls.cc, which reads the tensors and makes the call in native code; ctypes is
left for what is called once per program (and for kernel variants that a test forces).
"""
import ctypes as C

import torch

from . import _lib

EPI_ACC_S32, EPI_REQUANT_CPU, EPI_REQUANT_GPU, EPI_DEQUANT_F32 = 0, 1, 2, 3
# requant, then dequantize with the per-tensor output scale, in one epilogue
EPI_REQUANT_CPU_DEQUANT_F32, EPI_REQUANT_GPU_DEQUANT_F32 = 4, 5
EPI_REQUANT_FIXEDPOINT = 6
BIAS_NONE, BIAS_S32, BIAS_F32, BIAS_S8 = 0, 1, 2, 3
ROUND_HALF_AWAY_FROM_ZERO, ROUND_HALF_TO_EVEN = 0, 1

_BIAS_KIND = {torch.int32: BIAS_S32, torch.float32: BIAS_F32, torch.int8: BIAS_S8}
_OUT_DTYPE = {EPI_ACC_S32: torch.int32, EPI_REQUANT_CPU: torch.int8,
              EPI_REQUANT_GPU: torch.int8, EPI_DEQUANT_F32: torch.float32,
              EPI_REQUANT_CPU_DEQUANT_F32: torch.float32,
              EPI_REQUANT_GPU_DEQUANT_F32: torch.float32,
              EPI_REQUANT_FIXEDPOINT: torch.int8}


def _native():
    """The native callers; replaces itself by the loaded module's accessor on first use."""
    global _native
    mod = _lib.torch_calls()
    _native = lambda: mod  # noqa: E731
    return mod


def _ptr(t):
    return C.c_void_p(t.data_ptr()) if t is not None else None


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _need_cuda(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise ValueError("expected device tensors")


def _scale(t, device):
    if not torch.is_tensor(t):
        t = torch.tensor(t, dtype=torch.float32, device=device)
    return t.reshape(-1).contiguous().float()


def variant_names():
    """Names of the kernel variants a test can force (from the test-hooks library)."""
    L = _lib.hooks()
    return [L.dq8_qgemm_variant_name(i).decode() for i in range(L.dq8_qgemm_num_variants())]


def _view3(shape, axis):
    n = 1
    for s in shape:
        n *= s
    if axis is None:
        return 1, 1, n
    outer = 1
    for s in shape[:axis]:
        outer *= s
    inner = 1
    for s in shape[axis + 1:]:
        inner *= s
    return outer, shape[axis], inner


# quantized element types: name -> (kind of the C ABI, torch dtype that stores the bits)
QUANT_KINDS = {"int8": (0, torch.int8), "uint8": (1, torch.uint8), "int16": (2, torch.int16),
               "uint16": (3, torch.int16), "int32": (4, torch.int32), "uint32": (5, torch.int32)}


# (by torch dtype as well: a dict lookup per call)
_KINDS = {**QUANT_KINDS, **{getattr(torch, name): (kind, getattr(torch, name))
                            for name, (kind, _) in QUANT_KINDS.items() if hasattr(torch, name)}}


def quantize(x, scale, zero_point, axis=None, qmin=-128, qmax=127,
             round_mode=ROUND_HALF_TO_EVEN, dtype=torch.int8, out=None):
    """mhlo_disc.quantize on the GPU.  scale/zero_point: device tensors (f32 / i32); x: f32 or
    f16.  dtype: a torch dtype or one of the names in QUANT_KINDS -- the unsigned 16 / 32 bit
    types are returned in the signed torch dtype of the same width (same bits)."""
    if out is not None and not isinstance(dtype, str):
        dtype = out.dtype
    kind, store = _KINDS[dtype]
    return _native().quantize(x, scale, zero_point, axis, qmin, qmax, round_mode, kind, store, out)


def fake_quant(x, scale, zero_point, axis=None, qmin=-128, qmax=127,
               round_mode=ROUND_HALF_TO_EVEN, out=None):
    """dequantize(quantize(x)) in one pass: f32 -> f32, the same bits as the two calls."""
    return _native().fake_quant(x, scale, zero_point, axis, qmin, qmax, round_mode, out)


def minmax(x, min_io, max_io, axis=None, workspace=None):
    """Folds the minimum and maximum of `x` (device f32), per tensor (axis None) or per
    slice along `axis`, into the running values min_io / max_io (device f32, one entry or
    one per channel).  Returns (min_io, max_io)."""
    _native().minmax(x, min_io, max_io, axis, workspace)
    return min_io, max_io


def observe(x, min_io, max_io, symmetric, q_min, q_max, axis=None, fake_quant=False):
    """One observation step: minmax(x, min_io, max_io, axis), then the 8-bit scale and zero point
    of every channel from the running values and, if asked for, fake_quant(x) with them.  Returns
    (sound, scale, zero_point, fake-quantized x or None); `sound` is False when a channel's
    minimum is not at most its maximum (a NaN was observed).  x must not be empty."""
    return _native().observe(x, min_io, max_io, axis, symmetric, q_min, q_max, fake_quant)


def lut8(q, table, out=None):
    """out[i] = table[bit pattern of q[i]] for an int8 / uint8 device tensor; `table` is a
    256-entry device tensor of the output's 8-bit type."""
    return _native().lut8(q, table, out)


def weight_only_qgemm(x, w, scale, zero_points=None, bias=None, tp_b=True, out=None,
                      workspace=True):
    """out = x @ ((w - zero_points[:, None]) * scale[:, None]).T + bias for f16 / f32
    activations x [M,K] and 8-bit weights (uint8 or int8) w [N,K] (tp_b) or [K,N]; scale and
    bias have x's dtype, zero_points is int32.  workspace=False withholds the scratch that
    [K,N] weights are transposed into and that a launch split over k keeps its partial sums
    in; a uint8 tensor is used as that scratch."""
    return _native().weight_only_qgemm(x, w, scale, zero_points, bias, tp_b, out, workspace)


def weight_only_undo_compiler_layout(reordered_kn):
    """[K,N] uint8 bytes as the reference's compiler leaves a constant weight-only weight
    (`weight_should_be_reordered = false`) -> the dense [N,K] weight matrix."""
    _need_cuda(reordered_kn)
    if reordered_kn.dtype != torch.uint8 or reordered_kn.dim() != 2:
        raise TypeError("weight_only_undo_compiler_layout takes a uint8 [K,N] tensor")
    r = reordered_kn.contiguous()
    k, n = r.shape
    out = torch.empty((n, k), dtype=torch.uint8, device=r.device)
    st = _lib.lib().dq8_weight_only_undo_compiler_layout(_ptr(r), _ptr(out), k, n, _stream())
    _lib.check(st, "dq8_weight_only_undo_compiler_layout")
    return out


def activation_table(fn, s_in, z_in, s_out, z_out, in_dtype=torch.int8, out_dtype=torch.int8,
                     device="cuda"):
    """The table of  q -> quantize(fn(dequantize(q, s_in, z_in)), s_out, z_out)  for every
    8-bit q, built with the same dequantize / quantize kernels a chain of separate operators
    would run, so that  lut8(q, table)  equals that chain bit for bit.  s_*: one-element
    device f32 tensors, z_*: one-element device i32 tensors; fn: a torch elementwise function.
    Entry i belongs to the input whose bit pattern is i."""
    bits = torch.arange(256, dtype=torch.int16, device=device).to(torch.uint8)
    q = bits.view(in_dtype) if in_dtype != torch.uint8 else bits
    y = fn(dequantize(q, s_in, z_in))
    qmin, qmax = (-128, 127) if out_dtype == torch.int8 else (0, 255)
    return quantize(y, s_out, z_out, qmin=qmin, qmax=qmax, dtype=out_dtype)


def dequantize(q, scale, zero_point, axis=None, out=None, dtype=None):
    """mhlo_disc.dequantize on the GPU; dtype names the quantized type where q's torch dtype
    does not (the unsigned 16 / 32 bit types, see QUANT_KINDS)."""
    kind, _ = _KINDS[dtype if dtype is not None else q.dtype]
    return _native().dequantize(q, scale, zero_point, axis, kind, out)


def make_postops(residual=None, residual_scale=None, residual_zp=0, relu=False, out_scale=None,
                 out_zp=0, table=None):
    """dq8_postops_t for the operators fused behind a quantized GEMM / convolution; returns
    (struct, objects to keep alive).  residual: f32 or int8 device tensor of the output's
    shape (int8: with residual_scale, a one-element device tensor, and residual_zp);
    out_scale: one-element device tensor of the quantize that follows (int8 results);
    table: 256-entry int8 / uint8 device tensor."""
    po = _lib.PostOps()
    keep = []
    if residual is not None:
        if residual.stride(-1) != 1:
            residual = residual.contiguous()
        r2 = residual.reshape(-1, residual.shape[-1]) if residual.is_contiguous() else residual
        po.residual = r2.data_ptr()
        po.residual_kind = 1 if residual.dtype == torch.float32 else 2
        po.ldr = r2.stride(0)
        keep.append(r2)
        if residual_scale is not None:
            po.residual_scale = residual_scale.data_ptr()
            keep.append(residual_scale)
        po.residual_zp = int(residual_zp)
    po.relu = int(bool(relu))
    if out_scale is not None:
        po.out_scale = out_scale.data_ptr()
        keep.append(out_scale)
    po.out_zp = int(out_zp)
    if table is not None:
        po.table = table.data_ptr()
        keep.append(table)
    return po, keep


def qgemm(a, w, epilogue, sx=None, sw=None, so=None, bias=None, tp_a=False, tp_b=True,
          zx=0, zw=0, zo=0, variant=-1, out=None, post=None):
    """int8 GEMM with a fused epilogue.  a: [M,K] ([K,M] if tp_a); w: [N,K] if tp_b
    else [K,N]; scales are device f32 tensors with 1 or N entries."""
    if post is not None:
        if variant != -1:
            raise ValueError("fused operators go with the library's own choice of kernel")
        post = post[0] if isinstance(post, tuple) else post
    if variant == -1:
        return _native().qgemm(a, w, epilogue, sx, sw, so, bias, tp_a, tp_b, zx, zw, zo, out, post)
    # a forced kernel variant: the tests' entry point, in the test-hooks library
    _need_cuda(a, w, bias)
    L = _lib.hooks()
    # rows may be strided (leading dimension > row length); elements must be dense
    if a.dim() != 2 or a.stride(1) != 1:
        a = a.contiguous()
    if w.dim() != 2 or w.stride(1) != 1:
        w = w.contiguous()
    m, k = (a.shape[1], a.shape[0]) if tp_a else a.shape
    n = w.shape[0] if tp_b else w.shape[1]
    kw = w.shape[1] if tp_b else w.shape[0]
    if k != kw:
        raise ValueError("mismatch contraction dim")
    dev = a.device
    if out is None:
        out = torch.empty((m, n), dtype=_OUT_DTYPE[epilogue], device=dev)
    sx = _scale(sx, dev) if sx is not None else None
    sw = _scale(sw, dev) if sw is not None else None
    so = _scale(so, dev) if so is not None else None
    bias_kind = BIAS_NONE if bias is None else _BIAS_KIND[bias.dtype]
    ws_bytes = L.dq8_qgemm_workspace_bytes(m, n, k, int(tp_a), int(tp_b))
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev) if ws_bytes else None
    st = L.dq8_qgemm_variant(
        variant, _ptr(a), max(a.stride(0), a.shape[1]), _ptr(w), max(w.stride(0), w.shape[1]),
        _ptr(out), out.stride(0) if m else n, m, n, k, int(tp_a), int(tp_b), epilogue, _ptr(bias),
        bias_kind, _ptr(sx), sx.numel() if sx is not None else 0,
        _ptr(sw), sw.numel() if sw is not None else 0,
        _ptr(so), so.numel() if so is not None else 0, zx, zw, zo, _ptr(ws), ws_bytes, _stream())
    _lib.check(st, "dq8_qgemm", L)
    return out


def qlinear_f32_fused_max_rows(n, k):
    return int(_lib.lib().dq8_qlinear_f32_fused_max_rows(n, k))


def qlinear_f32(x, w, epilogue, sx, sw=None, so=None, bias=None, zo=0,
                round_mode=ROUND_HALF_TO_EVEN, out=None):
    """quantize(x; sx, zero point 0) -> qgemm(., w [N,K]) with the given epilogue, one launch,
    for a few rows of f32 activations x [M,K]; the same bits as quantize followed by qgemm."""
    return _native().qlinear_f32(x, w, epilogue, sx, sw, so, bias, zo, round_mode, out)


def attention(qkv, heads, scale=None, qkv_scale=None):
    """softmax(q k^T / sqrt(64)) v of a merged f32 projection [B, S, 3 * heads * 64] -> [B, S,
    heads * 64], f32 throughout; with a one-element device `scale` the result is quantized to int8
    in the same pass (the bits of quantize(., scale, 0) behind it).  With a one-element device
    `qkv_scale` the projection is int8, qkv_scale times which is what its products are of."""
    return _native().attention(qkv, heads, scale, qkv_scale)


def layer_norm(x, weight, bias, eps=1e-5, scale=None):
    """Layer normalisation over the last dimension (f32, up to 2048 columns, a multiple of 4);
    with a one-element device `scale` returns (y, quantize(y, scale, 0)) from one pass."""
    return _native().layer_norm(x, weight, bias, eps, scale)


def encoder_layer(h, heads, eps, operands):
    """A quantized encoder layer on h [B, S, 64 * heads] (f32): quantize, merged projection (int8), attention,
    output linear + h, layer norm, feed-forward linear with a 256-entry activation table, second
    feed-forward linear + the first norm, layer norm -- the calls above in this order, eight launches.
    operands: for the four linears in turn (int8 weights [N, K], f32 bias, input scale, weight scales,
    output scale), then the table, the norms' (weight, bias, weight, bias) and an int32 zero; all
    contiguous, one bias and weight scale per channel and one input and output scale.  None where an
    operand is of another form: then the calls one by one decide."""
    return _native().encoder_layer(h, heads, eps, operands)


NHWC_OHWI = (0, 3, 1, 2, 3, 0, 1, 2, 0, 3, 1, 2)


def qconv2d(x, w, padding, metadata, out_shape, epilogue, sx=None, sw=None, so=None,
            bias=None, zo=0, variant=-1, out=None, workspace=True, post=None):
    """int8 convolution; layouts/strides/dilations from the 17-entry ral_qconv
    metadata, padding = (top, bottom, left, right).  workspace=False withholds the scratch
    that keeps channel counts off a multiple of 16 on the MFMA kernels."""
    if post is not None:
        if variant != -1:
            raise ValueError("fused operators go with the library's own choice of kernel")
        post = post[0] if isinstance(post, tuple) else post
    if variant == -1:
        return _native().qconv2d(x, w, padding, metadata, out_shape, epilogue, sx, sw, so, bias, zo,
                                 out, workspace, post)
    # a forced kernel variant: the tests' entry point, in the test-hooks library
    _need_cuda(x, w, bias)
    L = _lib.hooks()
    x = x.contiguous()
    w = w.contiguous()
    dev = x.device
    if out is None:
        out = torch.empty(tuple(out_shape), dtype=_OUT_DTYPE[epilogue], device=dev)
    sx = _scale(sx, dev) if sx is not None else None
    sw = _scale(sw, dev) if sw is not None else None
    so = _scale(so, dev) if so is not None else None
    bias_kind = BIAS_NONE if bias is None else _BIAS_KIND[bias.dtype]
    i64x4 = C.c_int64 * 4
    md = (C.c_int32 * 17)(*metadata)
    ws_bytes = L.dq8_qconv2d_workspace_bytes_ex(i64x4(*x.shape), i64x4(*w.shape), i64x4(*out_shape), md) if workspace else 0
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev) if ws_bytes else None
    st = L.dq8_qconv2d_variant(
        variant, _ptr(x), i64x4(*x.shape), _ptr(w), i64x4(*w.shape), (C.c_int32 * 4)(*padding), md,
        _ptr(out), i64x4(*out_shape), epilogue, _ptr(bias), bias_kind, _ptr(sx), _ptr(sw),
        sw.numel() if sw is not None else 0, _ptr(so), zo, _ptr(ws), ws_bytes, _stream())
    _lib.check(st, "dq8_qconv2d", L)
    return out


def mfma_probe(a32, b32, a16, b16):
    d32 = torch.empty((32, 32), dtype=torch.int32, device=a32.device)
    d16 = torch.empty((16, 16), dtype=torch.int32, device=a32.device)
    st = _lib.hooks().dq8_mfma_probe(_ptr(a32), _ptr(b32), _ptr(d32), _ptr(a16), _ptr(b16),
                                     _ptr(d16), _stream())
    _lib.check(st, "dq8_mfma_probe", _lib.hooks())
    return d32, d16
