"""GPU parity tests of the raw kernel C ABI against the CPU oracle (bit-exact for
int32/int8 results; 1e-5 relative for f32 outputs)."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from bladedisc_amd import kernels
    return kernels


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def persistent_refuses(K, v, row, out_bytes):
    """Whether variant v is a persistent kernel that has no form for result rows of `row` elements
    of this size: they store 16 bytes at a time, the 256-row ones int8 alone."""
    name = K.variant_names()[v] if v >= 0 else ""
    return name.startswith("persist_") and (row * out_bytes % 16 != 0 or
                                            (out_bytes == 4 and name.startswith("persist_256x")))


def gemm_variants(K, k, row=16, out_bytes=1):
    """All variant ids of the GEMM that take result rows of `row` elements of this size."""
    return [i for i, nm in enumerate(K.variant_names())
            if not nm.startswith(("direct3x3_", "stream")) and not persistent_refuses(K, i, row, out_bytes)]


def make_scales(rng, n, per_channel=True):
    sx = np.float32(rng.uniform(0.01, 0.03))
    sw = rng.uniform(0.001, 0.05, n if per_channel else 1).astype(np.float32)
    return sx, sw


def pick_so(acc, sx, sw):
    """Output scale putting the results at about 40 LSB rms (few saturate)."""
    s = float(np.std(acc.astype(np.float64) * (float(sx) * sw.astype(np.float64).mean())))
    return np.float32(max(s, 1e-6) / 40.0)


# ------------------------------------------------------------------ MFMA layout
def test_mfma_operand_and_result_layouts(K):
    rng = np.random.default_rng(0)
    a = rng.integers(-128, 128, (32, 32), dtype=np.int8)   # row i, k contiguous
    b = rng.integers(-128, 128, (32, 32), dtype=np.int8)   # column j, k contiguous
    a16 = rng.integers(-128, 128, (16, 64), dtype=np.int8)
    b16 = rng.integers(-128, 128, (16, 64), dtype=np.int8)
    d32, d16 = K.mfma_probe(dev(a), dev(b), dev(a16), dev(b16))
    np.testing.assert_array_equal(host(d32), a.astype(np.int32) @ b.astype(np.int32).T)
    np.testing.assert_array_equal(host(d16), a16.astype(np.int32) @ b16.astype(np.int32).T)


# ------------------------------------------------------------------------ qgemm
SHAPES = [(1, 768, 768), (16, 768, 768), (64, 768, 768), (128, 3072, 768), (1000, 768, 3072),
          (257, 130, 64), (33, 36, 16), (300, 260, 1040), (512, 512, 512), (5, 7, 48),
          # contraction lengths that are not a multiple of 16: padded into the scratch
          (4, 71, 25), (300, 260, 1041), (1000, 768, 777), (64, 64, 1), (2048, 1024, 15)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_qgemm_acc_s32_all_variants(K, m, n, k):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    want, _ = O.gemm_s32_fast(a, w)
    da, dw = dev(a), dev(w)
    for v in gemm_variants(K, k, n, 4):
        got = host(K.qgemm(da, dw, K.EPI_ACC_S32, variant=v))
        np.testing.assert_array_equal(got, want, err_msg=K.variant_names()[v])
    np.testing.assert_array_equal(host(K.qgemm(da, dw, K.EPI_ACC_S32)), want)


@pytest.mark.parametrize("m,n,k", [(64, 768, 768), (1000, 768, 3072), (257, 130, 64), (4096, 768, 768)])
@pytest.mark.parametrize("bias", ["none", "s32", "f32"])
def test_qgemm_requant_cpu(K, m, n, k, bias):
    rng = np.random.default_rng(m + n + k + len(bias))
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc, _ = O.gemm_s32_fast(a, w)
    sx, sw = make_scales(rng, n)
    so = pick_so(acc, sx, sw)
    b32 = bias_t = None
    if bias == "s32":
        b32 = rng.integers(-200000, 200000, n).astype(np.int32)
        bias_t = dev(b32)
    elif bias == "f32":
        bf = (rng.standard_normal(n) * 10 * so).astype(np.float32)
        b32 = O.bias_f32_to_s32(bf, sx, sw)
        bias_t = dev(bf)
    want = O.requant_cpu(acc, sx, sw, so, b32=b32)
    for v in [-1] + gemm_variants(K, k, n):
        got = host(K.qgemm(dev(a), dev(w), K.EPI_REQUANT_CPU, sx=dev(np.array([sx])), sw=dev(sw),
                           so=dev(np.array([so])), bias=bias_t, variant=v))
        np.testing.assert_array_equal(got, want, err_msg="variant %d" % v)
    sat = np.mean((want == 127) | (want == -128))
    assert sat < 0.5, "degenerate test: %.2f saturated" % sat


@pytest.mark.parametrize("m,n,k", [
    (4133, 4112, 272),     # 17 x 17 tiles of 256 x 256: more tiles than compute units, not a multiple of 8
    (4133, 4109, 272),     # (result rows at any byte: no persistent form)
    (4096, 4304, 144),     # 16 x 17 = 272 tiles: dealt per XCD; two k tiles, the second ragged
    (4096, 4300, 144),     # (rows of 4-byte results alone on 16 bytes)
    (5000, 3840, 128),     # 20 x 20 tiles of 256 x 192 / 20 x 15 of 256 x 256; one k tile
    (16384, 1536, 400),    # three and four rounds of the two big tile shapes
])
def test_qgemm_persistent_variants_walk_many_tiles(K, m, n, k):
    """The persistent kernels with several output tiles per workgroup: ragged last tiles in
    M, N and K, tile counts that do and do not divide over the XCDs, all epilogue families
    (int8 with and without additive terms; int32 and f32 from the 128-row form, which alone has
    them), and the heuristic's own pick at these sizes -- bit-exact against the oracle."""
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc, _ = O.gemm_s32_fast(a, w)
    sx, sw = make_scales(rng, n)
    so = pick_so(acc, sx, sw)
    bf = (rng.standard_normal(n) * 10 * so).astype(np.float32)
    b32 = O.bias_f32_to_s32(bf, sx, sw)
    want_plain = O.requant_cpu(acc, sx, sw, so)
    want_bias = O.requant_cpu(acc, sx, sw, so, b32=b32, zo=3)
    want_f32 = O.dequant_acc(acc, sx, sw, bias=bf)
    da, dw = dev(a), dev(w)
    dsx, dsw, dso = dev(np.array([sx])), dev(sw), dev(np.array([so]))
    names = K.variant_names()
    persistent = [i for i, nm in enumerate(names) if nm.startswith("persist_")]
    assert len(persistent) == 3
    for v in [-1] + persistent:
        tag = names[v] if v >= 0 else "heuristic"
        if not persistent_refuses(K, v, n, 1):
            got = host(K.qgemm(da, dw, K.EPI_REQUANT_CPU, sx=dsx, sw=dsw, so=dso, variant=v))
            np.testing.assert_array_equal(got, want_plain, err_msg=tag)
            got = host(K.qgemm(da, dw, K.EPI_REQUANT_CPU, sx=dsx, sw=dsw, so=dso, bias=dev(bf), zo=3,
                               variant=v))
            np.testing.assert_array_equal(got, want_bias, err_msg=tag)
            got = host(K.qgemm(da, dw, K.EPI_REQUANT_GPU, sx=dsx, sw=dsw, so=dso, bias=dev(bf), variant=v))
            np.testing.assert_array_equal(got, O.requant_gpu(acc, sx, sw, so, bias_f32=bf), err_msg=tag)
        if persistent_refuses(K, v, n, 4):
            continue
        np.testing.assert_array_equal(host(K.qgemm(da, dw, K.EPI_ACC_S32, variant=v)), acc, err_msg=tag)
        got = host(K.qgemm(da, dw, K.EPI_DEQUANT_F32, sx=dsx, sw=dsw, bias=dev(bf), variant=v))
        assert np.array_equal(got.view(np.uint32), want_f32.view(np.uint32)), tag
        # requant -> dequantize in one epilogue (f32 result) and the E2 form with its f32 bias
        got = host(K.qgemm(da, dw, K.EPI_REQUANT_CPU_DEQUANT_F32, sx=dsx, sw=dsw, so=dso, bias=dev(bf),
                           zo=3, variant=v))
        want = O.dequantize(want_bias, np.array([so], np.float32), np.array([3], np.int32))
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), tag


def test_forced_persistent_variants_refuse_what_they_have_no_form_for(K):
    """A forced persistent kernel runs or says so: no other kernel in its place."""
    one = torch.ones(1, device="cuda")
    sc = dict(sx=one, sw=one, so=one)
    a = torch.zeros((300, 64), dtype=torch.int8, device="cuda")
    refused = 0
    for v, name in enumerate(K.variant_names()):
        if not name.startswith("persist_"):
            continue
        for n, epi, out_bytes in ((256, K.EPI_ACC_S32, 4), (256, K.EPI_DEQUANT_F32, 4), (256, K.EPI_REQUANT_CPU, 1),
                                  (264, K.EPI_REQUANT_GPU, 1), (258, K.EPI_REQUANT_CPU_DEQUANT_F32, 4)):
            w = torch.zeros((n, 64), dtype=torch.int8, device="cuda")
            kw = {} if epi == K.EPI_ACC_S32 else sc
            if persistent_refuses(K, v, n, out_bytes):
                refused += 1
                with pytest.raises(RuntimeError, match="persistent"):
                    K.qgemm(a, w, epi, variant=v, **kw)
            else:
                assert not K.qgemm(a, w, epi, variant=v, **kw).any()
    assert refused == 2 * 4 + 2


@pytest.mark.parametrize("m,n,k", [(64, 768, 768), (1000, 768, 3072), (257, 130, 64), (5, 7, 48),
                                   (4096, 768, 768), (300, 260, 1041)])
@pytest.mark.parametrize("bias", ["none", "s32"])
def test_qgemm_requant_fixedpoint(K, m, n, k, bias):
    """The integer output stage of the reference's AArch64 path (multiplier + shift) in every
    kernel variant, per-channel and per-tensor weight scales, with and without an output zero
    point, multipliers below and above one -- bit-exact against the oracle's restatement."""
    rng = np.random.default_rng(m + 5 * n + k + len(bias))
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc, _ = O.gemm_s32_fast(a, w)
    sx, sw = make_scales(rng, n)
    so = pick_so(acc, sx, sw)
    b32 = rng.integers(-200000, 200000, n).astype(np.int32) if bias == "s32" else None
    bias_t = dev(b32) if b32 is not None else None
    cases = [(sw, so, 0), (sw, so, -5), (sw[:1], so, 0),
             (sw, np.float32(so * 1e-5), 7)]          # multipliers above one: left shifts, saturation
    for swv, sov, zo in cases:
        want = O.requant_fixedpoint(acc, sx, swv, sov, b32=b32, zo=zo)
        for v in [-1] + gemm_variants(K, k):
            if K.variant_names()[v].startswith("persist_") and v >= 0:
                # (the persistent kernels leave this stage out and say so when forced)
                with pytest.raises(RuntimeError, match="persistent"):
                    K.qgemm(dev(a), dev(w), K.EPI_REQUANT_FIXEDPOINT, sx=dev(np.array([sx])),
                            sw=dev(swv), so=dev(np.array([sov], np.float32)), bias=bias_t, zo=zo,
                            variant=v)
                continue
            got = host(K.qgemm(dev(a), dev(w), K.EPI_REQUANT_FIXEDPOINT, sx=dev(np.array([sx])),
                               sw=dev(swv), so=dev(np.array([sov], np.float32)), bias=bias_t, zo=zo,
                               variant=v))
            np.testing.assert_array_equal(got, want, err_msg="variant %d zo %d" % (v, zo))
    want = O.requant_fixedpoint(acc, sx, sw, so, b32=b32)
    sat = np.mean((want == 127) | (want == -128))
    assert sat < 0.5, "degenerate test: %.2f saturated" % sat
    # it is a different rounding from the float stage, not the same numbers by another route
    other = O.requant_cpu(acc, sx, sw, so, b32=b32)
    assert np.max(np.abs(other.astype(np.int32) - want.astype(np.int32))) <= 1


@pytest.mark.parametrize("m,n,k", [(64, 768, 768), (1000, 768, 3072), (257, 132, 64), (5, 16, 48),
                                   (4096, 768, 768), (3072, 3072, 768), (300, 260, 96)])
def test_qgemm_fused_operators_equal_the_separate_ones(K, m, n, k):
    """Operators fused behind a quantized GEMM -- dequantize -> +residual (f32 or int8) ->
    ReLU -> quantize, dequantize -> +residual -> f32, and a 256-entry table on the int8
    result -- give the bits of the chain of separate library calls (qgemm, dq8_dequantize, an
    f32 add, a clamp at zero, dq8_quantize, dq8_lut8), for every epilogue family."""
    rng = np.random.default_rng(11 * m + n + k)
    a = dev(rng.integers(-128, 128, (m, k), dtype=np.int8))
    w = dev(rng.integers(-128, 128, (n, k), dtype=np.int8))
    acc, _ = O.gemm_s32_fast(host(a), host(w))
    sx, sw = make_scales(rng, n)
    so = pick_so(acc, sx, sw)
    dsx, dsw, dso = dev(np.array([sx])), dev(sw), dev(np.array([so], np.float32))
    bias = dev((rng.standard_normal(n) * 10 * so).astype(np.float32))
    b32 = dev(rng.integers(-100000, 100000, n).astype(np.int32))
    rf = dev((rng.standard_normal((m, n)) * 40 * so).astype(np.float32))
    rq = dev(rng.integers(-128, 128, (m, n), dtype=np.int8))
    rs, rz = dev(np.array([so * 1.7], np.float32)), 4
    s2, z2 = dev(np.array([so * 1.3], np.float32)), -7
    zero = torch.zeros(1, dtype=torch.int32, device="cuda")
    table = dev(rng.integers(-128, 128, 256, dtype=np.int8))

    def unfused(q, zo, resid, relu, requant):
        y = K.dequantize(q, dso, torch.full((1,), zo, dtype=torch.int32, device="cuda"))
        r = resid if resid.dtype == torch.float32 else \
            K.dequantize(resid, rs, torch.full((1,), rz, dtype=torch.int32, device="cuda"))
        t = y + r
        if relu:
            t = torch.where(t < 0, torch.zeros_like(t), t)
        if not requant:
            return t
        return K.quantize(t, s2, torch.full((1,), z2, dtype=torch.int32, device="cuda"))

    stages = [(K.EPI_REQUANT_CPU, K.EPI_REQUANT_CPU_DEQUANT_F32, bias, 3),
              (K.EPI_REQUANT_GPU, K.EPI_REQUANT_GPU_DEQUANT_F32, bias, 0),
              (K.EPI_REQUANT_FIXEDPOINT, None, b32, -2)]
    for epi, epi_f32, b, zo in stages:
        q = K.qgemm(a, w, epi, sx=dsx, sw=dsw, so=dso, bias=b, zo=zo)
        for resid in (rf, rq):
            for relu in (False, True):
                kw = dict(residual=resid, relu=relu)
                if resid.dtype == torch.int8:
                    kw.update(residual_scale=rs, residual_zp=rz)
                got = K.qgemm(a, w, epi, sx=dsx, sw=dsw, so=dso, bias=b, zo=zo,
                              post=K.make_postops(out_scale=s2, out_zp=z2, **kw))
                assert torch.equal(got, unfused(q, zo, resid, relu, True)), (epi, resid.dtype, relu)
                if epi_f32 is not None:
                    got = K.qgemm(a, w, epi_f32, sx=dsx, sw=dsw, so=dso, bias=b, zo=zo,
                                  post=K.make_postops(**kw))
                    want = unfused(q, zo, resid, relu, False)
                    assert torch.equal(got.view(torch.int32), want.view(torch.int32)), \
                        (epi_f32, resid.dtype, relu)
        got = K.qgemm(a, w, epi, sx=dsx, sw=dsw, so=dso, bias=b, zo=zo,
                      post=K.make_postops(table=table))
        assert torch.equal(got, K.lut8(q, table)), epi
    # what the API refuses
    with pytest.raises(RuntimeError, match="out_scale"):
        K.qgemm(a, w, K.EPI_REQUANT_CPU, sx=dsx, sw=dsw, so=dso, post=K.make_postops(residual=rf))
    with pytest.raises(RuntimeError, match="requantising"):
        K.qgemm(a, w, K.EPI_ACC_S32, post=K.make_postops(table=table))
    with pytest.raises(RuntimeError, match="no residual"):
        K.qgemm(a, w, K.EPI_REQUANT_CPU, sx=dsx, sw=dsw, so=dso,
                post=K.make_postops(table=table, residual=rf, out_scale=s2))
    assert zero.item() == 0


@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("bias", ["none", "f32", "s8"])
def test_qgemm_requant_gpu(K, per_channel, bias):
    m, n, k = 200, 384, 512
    rng = np.random.default_rng(17 + per_channel)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc, _ = O.gemm_s32_fast(a, w)
    ns = n if per_channel else 1
    sx = rng.uniform(0.01, 0.03, ns).astype(np.float32)
    sw = rng.uniform(0.001, 0.05, ns).astype(np.float32)
    so = (np.full(ns, pick_so(acc, sx.mean(), sw)) * rng.uniform(0.9, 1.1, ns)).astype(np.float32)
    bf = bi = bias_t = None
    if bias == "f32":
        bf = (rng.standard_normal(n) * 10).astype(np.float32)
        bias_t = dev(bf)
    elif bias == "s8":
        bi = rng.integers(-128, 128, n).astype(np.int8)
        bias_t = dev(bi)
    want = O.requant_gpu(acc, sx, sw, so, bias_f32=bf, bias_i8=bi)
    for v in [-1] + gemm_variants(K, k, n):
        got = host(K.qgemm(dev(a), dev(w), K.EPI_REQUANT_GPU, sx=dev(sx), sw=dev(sw), so=dev(so),
                           bias=bias_t, variant=v))
        np.testing.assert_array_equal(got, want, err_msg="variant %d" % v)


@pytest.mark.parametrize("m,n,k", [(64, 768, 768), (1000, 768, 3072), (257, 130, 64), (3072, 3072, 768),
                                   (5, 130, 784)])
@pytest.mark.parametrize("form", ["cpu_f32", "cpu_s32_zo", "gpu_s8", "gpu_none"])
def test_qgemm_requant_then_dequantize_in_one_epilogue(K, m, n, k, form):
    """Epilogues 4 / 5: the f32 result must equal, bit for bit, dequantize applied to the int8
    result of the requant epilogue -- against the oracle's two functions and against the two
    separate GPU kernels."""
    rng = np.random.default_rng(m * 7 + n + k + len(form))
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc, _ = O.gemm_s32_fast(a, w)
    sx, sw = make_scales(rng, n)
    so = pick_so(acc, sx, sw)
    zo = 0
    t = lambda v: dev(np.array([v], np.float32))
    if form.startswith("cpu"):
        epi, fused = K.EPI_REQUANT_CPU, K.EPI_REQUANT_CPU_DEQUANT_F32
        if form == "cpu_f32":
            bf = (rng.standard_normal(n) * 10 * so).astype(np.float32)
            bias_t, b32 = dev(bf), O.bias_f32_to_s32(bf, sx, sw)
        else:
            b32 = rng.integers(-200000, 200000, n).astype(np.int32)
            bias_t, zo = dev(b32), 5
        q_want = O.requant_cpu(acc, sx, sw, so, b32=b32, zo=zo)
    else:
        epi, fused = K.EPI_REQUANT_GPU, K.EPI_REQUANT_GPU_DEQUANT_F32
        bi = rng.integers(-128, 128, n).astype(np.int8) if form == "gpu_s8" else None
        bias_t = dev(bi) if bi is not None else None
        q_want = O.requant_gpu(acc, np.array([sx], np.float32), sw, np.array([so], np.float32),
                               bias_i8=bi)
    want = O.dequantize(q_want, np.array([so], np.float32), np.array([zo], np.int32))
    sov, zov = t(so), dev(np.array([zo], np.int32))
    for v in [-1] + gemm_variants(K, k, n):
        f32_v = -1 if persistent_refuses(K, v, n, 4) else v
        got = K.qgemm(dev(a), dev(w), fused, sx=t(sx), sw=dev(sw), so=sov, bias=bias_t, zo=zo,
                      variant=f32_v)
        assert got.dtype == torch.float32
        two = K.dequantize(K.qgemm(dev(a), dev(w), epi, sx=t(sx), sw=dev(sw), so=sov, bias=bias_t,
                                   zo=zo, variant=v), sov, zov)
        assert torch.equal(got, two), "variant %d" % v
        assert np.array_equal(host(got).view(np.uint32), want.view(np.uint32)), "variant %d" % v
    # a per-channel output scale is refused
    with pytest.raises(RuntimeError, match="per-tensor"):
        K.qgemm(dev(a), dev(w), fused, sx=t(sx), sw=dev(sw), so=dev(np.full(n, so, np.float32)),
                bias=bias_t, zo=zo)


def test_qgemm_dequant_f32(K):
    m, n, k = 64, 768, 768
    rng = np.random.default_rng(5)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc, _ = O.gemm_s32_fast(a, w)
    sx, sw = make_scales(rng, n)
    bias = rng.standard_normal(n).astype(np.float32)
    want = O.dequant_acc(acc, sx, sw, bias)
    exact = acc.astype(np.float64) * (np.float64(sx) * sw.astype(np.float64)) + bias
    for v in [-1] + gemm_variants(K, k, n, 4):
        got = host(K.qgemm(dev(a), dev(w), K.EPI_DEQUANT_F32, sx=dev(np.array([sx])), sw=dev(sw),
                           bias=dev(bias), variant=v))
        np.testing.assert_array_equal(got, want)
        # tolerance stated by the task for dequantized outputs: 1e-5 relative
        np.testing.assert_allclose(got, exact, rtol=1e-5, atol=1e-5 * np.abs(exact).max())


@pytest.mark.parametrize("tp_a,tp_b", [(0, 0), (1, 0), (1, 1)])
def test_qgemm_transposed_operands(K, tp_a, tp_b):
    m, n, k = 96, 200, 320
    rng = np.random.default_rng(31)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (k, n), dtype=np.int8)
    want = O.gemm_s32(a, w)
    a_in = a.T.copy() if tp_a else a
    w_in = w.T.copy() if tp_b else w
    for v in [-1, 0, 2]:
        got = host(K.qgemm(dev(a_in), dev(w_in), K.EPI_ACC_S32, tp_a=bool(tp_a), tp_b=bool(tp_b),
                           variant=v))
        np.testing.assert_array_equal(got, want)


def test_qgemm_ragged_k_stays_on_the_mfma_kernels(K):
    """K % 16 != 0: with the scratch dq8_qgemm_workspace_bytes asks for, the operands are
    padded and the MFMA kernels run (every layout, zero points, every epilogue); the result
    is the oracle's, and it is not the generic kernel's speed."""
    import time
    rng = np.random.default_rng(77)
    m, n, k = 1000, 520, 777
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    for tp_a, tp_b, zx, zw in [(0, 1, 0, 0), (1, 0, 0, 0), (0, 0, 5, 0), (1, 1, -9, 4)]:
        acc = O.gemm_s32(a, w, tp_b=True, zx=zx, zw=zw)
        a_in = np.ascontiguousarray(a.T) if tp_a else a
        w_in = w if tp_b else np.ascontiguousarray(w.T)
        kw = dict(tp_a=bool(tp_a), tp_b=bool(tp_b), zx=zx, zw=zw)
        np.testing.assert_array_equal(host(K.qgemm(dev(a_in), dev(w_in), K.EPI_ACC_S32, **kw)), acc)
        sx, sw = make_scales(rng, n)
        so = pick_so(acc, sx, sw)
        bias = (rng.standard_normal(n) * 3).astype(np.float32)
        want = O.requant_cpu(acc, sx, sw, so, b32=O.bias_f32_to_s32(bias, sx, sw))
        got = host(K.qgemm(dev(a_in), dev(w_in), K.EPI_REQUANT_CPU, sx=dev(np.array([sx])),
                           sw=dev(sw), so=dev(np.array([so])), bias=dev(bias), **kw))
        np.testing.assert_array_equal(got, want)
    # speed: 4096 x 4096 x 4095 would take the generic kernel seconds
    big = 4096
    ab = torch.randint(-128, 128, (big, big - 1), dtype=torch.int8, device="cuda")
    wb = torch.randint(-128, 128, (big, big - 1), dtype=torch.int8, device="cuda")
    out = K.qgemm(ab, wb, K.EPI_ACC_S32)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    out = K.qgemm(ab, wb, K.EPI_ACC_S32)
    torch.cuda.synchronize()
    assert time.perf_counter() - t0 < 0.01
    rows = [0, 1234, big - 1]
    want = O.gemm_s32(ab[rows].cpu().numpy(), wb.cpu().numpy(), tp_b=True)
    np.testing.assert_array_equal(out[rows].cpu().numpy(), want)


def test_qgemm_zero_points_generic(K):
    m, n, k = 17, 19, 23
    rng = np.random.default_rng(3)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    want = O.gemm_s32(a, w, tp_b=True, zx=3, zw=-4)
    got = host(K.qgemm(dev(a), dev(w), K.EPI_ACC_S32, zx=3, zw=-4))
    np.testing.assert_array_equal(got, want)
    with pytest.raises(RuntimeError):
        K.qgemm(dev(a), dev(w), K.EPI_ACC_S32, zx=3, variant=2)


@pytest.mark.parametrize("m,n,k,tp_a,tp_b,zx,zw", [
    (64, 768, 768, 0, 1, 7, 0), (300, 130, 400, 0, 1, -128, 0), (33, 48, 64, 0, 1, 5, -3),
    (256, 512, 1040, 0, 0, 100, 0), (100, 96, 128, 1, 1, 127, 2), (1, 768, 3072, 0, 1, 11, 0),
    (1000, 768, 768, 0, 1, -77, 9),
    # one shape per pipelined tile: 256x256 and 128x128 on eight waves, 256x64, 64x64 with K split
    (4096, 2560, 128, 0, 1, 9, -4), (2048, 2048, 256, 0, 1, -128, 127), (16384, 64, 128, 0, 1, 3, 1),
    (256, 256, 2048, 0, 1, 100, -100), (4100, 2570, 4096, 0, 1, 1, 0),
])
def test_qgemm_zero_points_on_the_mfma_path(K, m, n, k, tp_a, tp_b, zx, zw):
    """Asymmetric operands stay on the MFMA kernels when the caller provides the scratch for
    the correction vectors (the accumulators start at them): every epilogue equals the oracle's direct sum of (a - zx)(w - zw);
    without the scratch the generic kernel gives the same result."""
    rng = np.random.default_rng(m + n + k + zx)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc = O.gemm_s32(a, w, tp_b=True, zx=zx, zw=zw)
    a_in = np.ascontiguousarray(a.T) if tp_a else a
    w_in = w if tp_b else np.ascontiguousarray(w.T)
    kw = dict(tp_a=bool(tp_a), tp_b=bool(tp_b), zx=zx, zw=zw)
    got = host(K.qgemm(dev(a_in), dev(w_in), K.EPI_ACC_S32, **kw))
    np.testing.assert_array_equal(got, acc)
    got0 = host(K.qgemm(dev(a_in), dev(w_in), K.EPI_ACC_S32, variant=0, **kw))   # generic
    np.testing.assert_array_equal(got0, acc)
    sx, sw = make_scales(rng, n)
    so = pick_so(acc, sx, sw)
    bias = (rng.standard_normal(n) * 3).astype(np.float32)
    dsx, dsw, dso = dev(np.array([sx])), dev(sw), dev(np.array([so]))
    b32 = O.bias_f32_to_s32(bias, sx, sw)
    want = O.requant_cpu(acc, sx, sw, so, b32=b32, zo=5)
    got = host(K.qgemm(dev(a_in), dev(w_in), K.EPI_REQUANT_CPU, sx=dsx, sw=dsw, so=dso,
                       bias=dev(bias), zo=5, **kw))
    np.testing.assert_array_equal(got, want)
    want = O.requant_gpu(acc, sx, sw, so, bias_f32=bias)
    got = host(K.qgemm(dev(a_in), dev(w_in), K.EPI_REQUANT_GPU, sx=dsx, sw=dsw, so=dso,
                       bias=dev(bias), **kw))
    np.testing.assert_array_equal(got, want)
    want = O.dequant_acc(acc, sx, sw, bias=bias)
    got = host(K.qgemm(dev(a_in), dev(w_in), K.EPI_DEQUANT_F32, sx=dsx, sw=dsw, bias=dev(bias), **kw))
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-6)


def test_qgemm_zero_points_full_size_property(K):
    """4096^3 with an input zero point: the result equals the symmetric result of
    the shifted problem computed another way -- acc(a - zx, w) = acc(a, w) - zx * colsum(w)
    -- with both sides from the GPU in int32 and the column sums from numpy."""
    n = 4096
    g = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randint(-128, 128, (n, n), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-128, 128, (n, n), dtype=torch.int8, device="cuda", generator=g)
    sym = K.qgemm(a, w, K.EPI_ACC_S32)
    asym = K.qgemm(a, w, K.EPI_ACC_S32, zx=37)
    colsum = w.to(torch.int32).sum(dim=1)
    assert torch.equal(asym, sym - 37 * colsum[None, :])


def test_qgemm_known_answers(K, golden):
    for case in golden["qgemm"]:
        m, k, n = case["m"], case["k"], case["n"]
        qx = np.full((m, k), case["qx"], np.int8)
        qw = np.full((k, n), case["qw"], np.int8)   # [K,N] as the CPU callers hand it
        sw = np.full(n if case["per_channel"] else 1, case["sw"], np.float32)
        out = host(K.qgemm(dev(qx), dev(qw), K.EPI_REQUANT_CPU, tp_b=False,
                           sx=dev(np.array([case["sx"]], np.float32)), sw=dev(sw),
                           so=dev(np.array([case["so"]], np.float32))))
        assert (out == case["q_out"]).all(), case["src"]
        f = host(K.dequantize(dev(out), dev(np.array([case["so"]], np.float32)),
                              dev(np.array([0], np.int32))))
        assert (f == case["expect_f32"]).all()


def test_qgemm_empty_and_k0(K):
    a = torch.empty((0, 64), dtype=torch.int8, device="cuda")
    w = torch.zeros((32, 64), dtype=torch.int8, device="cuda")
    assert K.qgemm(a, w, K.EPI_ACC_S32).shape == (0, 32)
    a = torch.empty((8, 0), dtype=torch.int8, device="cuda")
    w = torch.empty((32, 0), dtype=torch.int8, device="cuda")
    out = host(K.qgemm(a, w, K.EPI_ACC_S32))
    assert out.shape == (8, 32) and (out == 0).all()


def test_qgemm_output_zero_point_and_saturation(K):
    acc_vals = np.array([[0, 1000, -1000, 127 * 127 * 64]], np.int32)
    a = np.zeros((1, 64), np.int8)
    w = np.zeros((4, 64), np.int8)
    a[0, :] = 127
    w[1, :16] = 1; w[1, 16] = -16 + 8  # noqa: E702
    # simpler: check against the oracle on random data with zo != 0
    rng = np.random.default_rng(8)
    a = rng.integers(-128, 128, (40, 64), dtype=np.int8)
    w = rng.integers(-128, 128, (52, 64), dtype=np.int8)
    acc = O.gemm_s32(a, w, tp_b=True)
    sx, sw = np.float32(0.02), rng.uniform(0.001, 0.05, 52).astype(np.float32)
    so = np.float32(0.05)   # small: many values saturate on both sides
    want = O.requant_cpu(acc, sx, sw, so, zo=7)
    got = host(K.qgemm(dev(a), dev(w), K.EPI_REQUANT_CPU, sx=dev(np.array([sx])), sw=dev(sw),
                       so=dev(np.array([so])), zo=7))
    np.testing.assert_array_equal(got, want)
    assert (want == 127).any() and (want == -128).any()
    del acc_vals


# --------------------------------------------------------------- quantize/dequant
@pytest.mark.parametrize("shape,axis", [((1000, 768), None), ((64, 768), 1), ((768, 768), 0),
                                        ((4, 56, 56, 64), 3), ((3, 5, 7), 1), ((1001,), None),
                                        ((130, 260), 1), ((2, 6, 10), 0), ((4096, 4096), 1)])
@pytest.mark.parametrize("round_mode", [0, 1])
def test_quantize_dequantize_parity(K, shape, axis, round_mode):
    rng = np.random.default_rng(len(shape) * 100 + (axis or 0))
    x = (rng.standard_normal(shape) * 2).astype(np.float32)
    flat = x.reshape(-1)
    flat[: min(64, flat.size)] = (np.arange(min(64, flat.size)) - 32 + 0.5) * 0.05  # ties
    n = 1 if axis is None else shape[axis]
    scale = rng.uniform(0.02, 0.08, n).astype(np.float32)
    scale[0] = 0.05
    zp = rng.integers(-3, 4, n).astype(np.int32)
    want = O.quantize(x, scale, zp, axis=axis, round_mode=round_mode)
    got = host(K.quantize(dev(x), dev(scale), dev(zp), axis=axis, round_mode=round_mode))
    np.testing.assert_array_equal(got, want)
    want_f = O.dequantize(want, scale, zp, axis=axis)
    got_f = host(K.dequantize(dev(want), dev(scale), dev(zp), axis=axis))
    np.testing.assert_array_equal(got_f, want_f)


@pytest.mark.parametrize("shape,axis", [((1000, 768), None), ((1003,), None), ((64, 768), 1), ((768, 768), 0),
                                        ((2, 3, 4, 5), 1), ((32, 8, 8, 64), 3), ((33, 52), 1), ((5, 7), 1)])
@pytest.mark.parametrize("round_mode", [0, 1])
@pytest.mark.parametrize("unsigned", [False, True])
def test_fake_quant_equals_quantize_then_dequantize(K, shape, axis, round_mode, unsigned):
    """dq8_fake_quant against the oracle's quantize -> dequantize and against the two GPU
    kernels, bit for bit (ties, saturation, non-zero zero points, in place)."""
    rng = np.random.default_rng(len(shape) * 31 + shape[0] + round_mode + 2 * unsigned)
    x = (rng.standard_normal(shape) * 3).astype(np.float32)
    flat = x.reshape(-1)
    flat[::7] = np.round(flat[::7] * 4) / 8          # plenty of exact halves after scaling by 1/0.125
    flat[::11] = 1e9
    nq = shape[axis] if axis is not None else 1
    scale = np.full(nq, 0.125, np.float32) if nq == 1 else rng.choice([0.125, 0.25, 0.1], nq).astype(np.float32)
    zp = rng.integers(-10, 11, nq).astype(np.int32) + (128 if unsigned else 0)
    qmin, qmax = (0, 255) if unsigned else (-128, 127)
    dt = np.uint8 if unsigned else np.int8
    want = O.dequantize(O.quantize(x, scale, zp, axis=axis, qmin=qmin, qmax=qmax,
                                   round_mode=round_mode, dtype=dt), scale, zp, axis=axis)
    dx, ds, dz = dev(x), dev(scale), dev(zp)
    got = K.fake_quant(dx, ds, dz, axis=axis, qmin=qmin, qmax=qmax, round_mode=round_mode)
    assert np.array_equal(host(got).view(np.uint32), want.view(np.uint32))
    two = K.dequantize(K.quantize(dx, ds, dz, axis=axis, qmin=qmin, qmax=qmax, round_mode=round_mode,
                                  dtype=torch.uint8 if unsigned else torch.int8), ds, dz, axis=axis)
    assert torch.equal(got.view(torch.int32), two.view(torch.int32))
    K.fake_quant(dx, ds, dz, axis=axis, qmin=qmin, qmax=qmax, round_mode=round_mode, out=dx)   # in place
    assert torch.equal(dx.view(torch.int32), got.view(torch.int32))
    # idempotent on its own output
    again = K.fake_quant(got, ds, dz, axis=axis, qmin=qmin, qmax=qmax, round_mode=round_mode)
    assert torch.equal(again, got)


def test_quantize_golden_vectors(K, golden):
    """Every vector of disc-fold-quantize.mlir, all six quantized types (the unsigned 16 / 32
    bit results come back as bits in the signed torch dtype of the same width)."""
    seen = set()
    for case in golden["quantize_fold"]:
        x = np.array(case["x"], np.float32)
        got = host(K.quantize(dev(x), dev(np.array(case["scale"], np.float32)),
                              dev(np.array(case["zp"], np.int32)), axis=case["axis"],
                              qmin=case["qmin"], qmax=case["qmax"], round_mode=case["round_mode"],
                              dtype=case["dtype"]))
        np.testing.assert_array_equal(got.view(case["dtype"]), np.array(case["expect"], case["dtype"]),
                                      err_msg=case["src"])
        seen.add(case["dtype"])
    assert seen == {"int8", "uint8", "int16", "uint16", "int32", "uint32"}


@pytest.mark.parametrize("name", ["int16", "uint16", "int32", "uint32"])
@pytest.mark.parametrize("axis", [None, 0, 1])
def test_quantize_dequantize_wide_types(K, name, axis):
    """16- and 32-bit quantized types against the oracle: values that land inside the range,
    on both limits and beyond them (the conversion of the clamped value saturates), both
    rounding modes, per tensor and per channel; dequantize back."""
    rng = np.random.default_rng(len(name) + (axis or 0) * 7)
    npdt = np.dtype(name)
    info = np.iinfo(npdt)
    shape = (37, 24)
    nq = 1 if axis is None else shape[axis]
    scale = rng.uniform(0.001, 0.01, nq).astype(np.float32)
    zp = rng.integers(-50, 50, nq).astype(np.int32) if info.min < 0 else rng.integers(0, 100, nq).astype(np.int32)
    span = float(info.max) * float(scale.mean())
    x = (rng.standard_normal(shape) * span * 0.6).astype(np.float32)
    x[0, :4] = [span * 4, -span * 4, span, -span]
    for rm in (0, 1):
        want = O.quantize(x, scale, zp, axis=axis, qmin=int(info.min), qmax=int(info.max),
                          round_mode=rm, dtype=npdt)
        got = K.quantize(dev(x), dev(scale), dev(zp), axis=axis, qmin=int(info.min),
                         qmax=int(info.max), round_mode=rm, dtype=name)
        np.testing.assert_array_equal(host(got).view(npdt), want)
        assert (want == info.max).any() and (want == info.min).any()
    back = K.dequantize(got, dev(scale), dev(zp), axis=axis, dtype=name)
    want_f = O.dequantize(want, scale, zp, axis=axis)
    assert np.array_equal(host(back).view(np.uint32), want_f.view(np.uint32))


@pytest.mark.parametrize("name", ["int8", "uint8", "int16"])
def test_quantize_f16_input_is_the_f32_path_on_the_widened_values(K, name):
    """Half-precision input (an extension: the reference's lowering takes f32 only) is widened
    exactly and then quantized by the f32 steps."""
    rng = np.random.default_rng(3)
    npdt = np.dtype(name)
    info = np.iinfo(npdt)
    x16 = (rng.standard_normal((50, 33)) * 3).astype(np.float16)
    scale = rng.uniform(0.01, 0.05, 33).astype(np.float32)
    zp = np.full(33, int((int(info.min) + int(info.max) + 1) // 2), np.int32)
    want = O.quantize(x16.astype(np.float32), scale, zp, axis=1, qmin=int(info.min),
                      qmax=int(info.max), dtype=npdt)
    got = K.quantize(dev(x16), dev(scale), dev(zp), axis=1, qmin=int(info.min), qmax=int(info.max),
                     dtype=name)
    np.testing.assert_array_equal(host(got).view(npdt), want)


def test_quantize_unaligned_and_uint8(K):
    rng = np.random.default_rng(2)
    x = (rng.standard_normal(4099) * 50).astype(np.float32)
    base = dev(np.concatenate([[0.0], x]).astype(np.float32))
    xv = base[1:]                                      # 4-byte aligned only
    scale, zp = np.array([0.5], np.float32), np.array([128], np.int32)
    want = O.quantize(x, scale, zp, qmin=0, qmax=255, dtype=np.uint8)
    out = torch.empty(4099, dtype=torch.uint8, device="cuda")
    K.quantize(xv, dev(scale), dev(zp), qmin=0, qmax=255, dtype=torch.uint8, out=out)
    np.testing.assert_array_equal(host(out), want)
    got_f = host(K.dequantize(dev(want), dev(scale), dev(zp)))
    np.testing.assert_array_equal(got_f, O.dequantize(want, scale, zp))


def test_quantize_empty(K):
    x = torch.empty((0, 8), device="cuda")
    s = torch.ones(1, device="cuda")
    z = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert K.quantize(x, s, z).shape == (0, 8)


# ------------------------------------------------------------------------- table
@pytest.mark.parametrize("n", [0, 1, 15, 16, 17, 4099, 1 << 20])
def test_lut8_matches_numpy_take(K, n):
    rng = np.random.default_rng(n)
    table = rng.integers(-128, 128, 256, dtype=np.int8)
    q = rng.integers(-128, 128, n, dtype=np.int8)
    want = table[q.view(np.uint8)]
    got = K.lut8(dev(q), dev(table))
    np.testing.assert_array_equal(host(got), want)
    if n > 20:
        base = dev(np.concatenate([[0], q]).astype(np.int8))
        view = base[1:]                                      # 1-byte aligned only
        np.testing.assert_array_equal(host(K.lut8(view, dev(table))), want)
        buf = dev(q)
        K.lut8(buf, dev(table), out=buf)                     # in place
        np.testing.assert_array_equal(host(buf), want)
    u = rng.integers(0, 256, max(n, 1), dtype=np.uint8)
    tu = rng.integers(0, 256, 256, dtype=np.uint8)
    np.testing.assert_array_equal(host(K.lut8(dev(u), dev(tu))), tu[u])


def test_activation_table_equals_the_operator_chain(K):
    """table[q] = quantize(f(dequantize(q))) built from the kernels themselves: a lookup
    equals running the three operators, for an asymmetric input and output."""
    rng = np.random.default_rng(2)
    q = dev(rng.integers(-128, 128, (300, 77), dtype=np.int8))
    s_in, z_in = dev(np.array([0.037], np.float32)), dev(np.array([-11], np.int32))
    s_out, z_out = dev(np.array([0.021], np.float32)), dev(np.array([7], np.int32))
    for fn in (torch.nn.functional.gelu, torch.tanh, torch.relu):
        table = K.activation_table(fn, s_in, z_in, s_out, z_out)
        chain = K.quantize(fn(K.dequantize(q, s_in, z_in)), s_out, z_out)
        assert torch.equal(K.lut8(q, table), chain)
        # and the oracle's view of it for one function with exact float32 semantics
    table = host(K.activation_table(torch.relu, s_in, z_in, s_out, z_out))
    allq = np.arange(256, dtype=np.uint8).view(np.int8)
    deq = O.dequantize(allq, np.float32(0.037), np.array([-11], np.int32))
    want = O.quantize(np.maximum(deq, 0), np.float32(0.021), np.array([7], np.int32))
    np.testing.assert_array_equal(table, want)


def test_qgemm_library_choice_on_random_shapes(K):
    """Seeded sweep over what decides the kernel of a GEMM -- rows from one to 16384, contraction
    lengths and channel counts that are and are not multiples of the tiles, transposed operands,
    zero points, every epilogue and bias kind: whatever the library picks gives the bytes
    (the floats, to 1e-6 relative) of the generic kernel, which the tests above pin to the
    oracle."""
    rng = np.random.default_rng(20260702)
    gen = K.variant_names().index("generic")
    done = 0
    for case in range(400):
        r = rng.random()
        if r < 0.5:
            m = int(rng.integers(1, 300))
            k = int(rng.choice([64, 128, 768, 1024, 3072, 4096, int(rng.integers(1, 3000))]))
            n = int(rng.choice([16, 64, 768, 3072, 4096, int(rng.integers(1, 2000))]))
        elif r < 0.92:
            m = int(rng.integers(300, 5000))
            k = int(rng.choice([128, 256, 768, 2304, int(rng.integers(1, 1500))]))
            n = int(rng.choice([64, 256, 768, 1024, 3072, int(rng.integers(1, 1500))]))
        else:
            m, k, n = int(rng.choice([8192, 16384, 12000])), int(rng.choice([768, 512])), int(rng.choice([768, 3072, 1000]))
        tp_b, tp_a = bool(rng.random() < 0.8), bool(rng.random() < 0.1)
        a = dev(rng.integers(-128, 128, (k, m) if tp_a else (m, k), dtype=np.int8))
        w = dev(rng.integers(-128, 128, (n, k) if tp_b else (k, n), dtype=np.int8))
        epi = int(rng.choice([K.EPI_ACC_S32, K.EPI_REQUANT_CPU, K.EPI_REQUANT_CPU, K.EPI_REQUANT_GPU, K.EPI_REQUANT_GPU,
                              K.EPI_DEQUANT_F32, K.EPI_REQUANT_CPU_DEQUANT_F32, K.EPI_REQUANT_GPU_DEQUANT_F32]))
        kw = dict(tp_a=tp_a, tp_b=tp_b)
        so = np.float32(0.02 * 0.025 * 74.0 * 74.0 * np.sqrt(k) / 40.0)
        if epi != K.EPI_ACC_S32:
            kw.update(sx=dev(np.array([0.02], np.float32)), so=dev(np.array([so])),
                      sw=dev(rng.uniform(0.001, 0.05, n if rng.random() < 0.8 else 1).astype(np.float32)))
        bk = int(rng.integers(0, 3))
        cpu_kind = epi in (K.EPI_REQUANT_CPU, K.EPI_REQUANT_CPU_DEQUANT_F32)
        gpu_kind = epi in (K.EPI_REQUANT_GPU, K.EPI_REQUANT_GPU_DEQUANT_F32)
        if cpu_kind and bk == 1:
            kw.update(bias=dev((rng.standard_normal(n) * 3 * so).astype(np.float32)))
        if cpu_kind and bk == 2:
            kw.update(bias=dev(rng.integers(-100000, 100000, n).astype(np.int32)))
        if gpu_kind and bk == 1:
            kw.update(bias=dev((rng.standard_normal(n) * 30).astype(np.float32)))
        if gpu_kind and bk == 2:
            kw.update(bias=dev(rng.integers(-128, 128, n, dtype=np.int8)))
        if epi == K.EPI_DEQUANT_F32 and bk:
            kw.update(bias=dev(rng.standard_normal(n).astype(np.float32)))
        kw.update(zx=int(rng.integers(-5, 5)) if rng.random() < 0.15 else 0,
                  zw=int(rng.integers(-5, 5)) if rng.random() < 0.1 else 0,
                  zo=int(rng.integers(-10, 10)) if epi == K.EPI_REQUANT_CPU else 0)
        got = K.qgemm(a, w, epi, **kw)
        want = K.qgemm(a, w, epi, variant=gen, **kw)
        tag = "case %d: %dx%dx%d, epilogue %d, bias kind %d, transposes %d %d, zero points %d %d %d" % (
            case, m, k, n, epi, bk, tp_a, tp_b, kw["zx"], kw["zw"], kw["zo"])
        if got.dtype == torch.float32:
            assert torch.allclose(got, want, rtol=1e-6, atol=0), tag
        else:
            assert torch.equal(got, want), tag
        done += 1
    assert done == 400


# ------------------------------------------------------------------------- conv
CONVS = [  # nb, h, w, ci, co, k, stride, pad, dil
    (2, 30, 30, 3, 64, 7, 2, 3, 1),      # an RGB first layer: channels padded into scratch
    (1, 9, 9, 20, 24, 3, 1, 1, 1),
    (2, 14, 14, 64, 64, 3, 1, 1, 1),
    (2, 9, 11, 32, 48, 3, 2, 1, 1),
    (1, 8, 8, 16, 16, 3, 1, 2, 2),
    (3, 7, 7, 256, 128, 1, 1, 0, 1),
    (2, 6, 6, 5, 6, 3, 1, 1, 1),      # Ci % 16 != 0 -> generic kernel
    (4, 28, 28, 64, 64, 3, 1, 1, 1),  # K = 576: a partial last k tile, several tiles of rows
    (2, 15, 13, 48, 80, 3, 2, 1, 2),  # ragged everything, K = 432
    # the direct 3x3 kernels: every channel count they take, images of one tile and of
    # several with a ragged last one, ragged Co, no / one / two pixels of padding
    (3, 20, 18, 32, 40, 3, 1, 1, 1),
    (2, 30, 30, 128, 136, 3, 1, 1, 1),
    (2, 12, 10, 256, 64, 3, 1, 0, 1),
    (1, 33, 17, 64, 200, 3, 1, 2, 1),
    (1, 36, 36, 256, 64, 3, 1, 1, 1),  # a patch of 107 KiB: LDS addresses beyond 128 KiB
    (1, 6, 150, 64, 64, 3, 1, 1, 1),   # a wide image: tiles of 256 pixels span 2-3 rows
    # 1 x 1 filters with a stride: the library runs them as a GEMM over the pixels they read
    (3, 14, 14, 256, 512, 1, 2, 0, 1),
    (2, 9, 11, 48, 80, 1, 2, 0, 1),    # odd image sizes, K = 48, ragged Co
    (5, 28, 28, 128, 256, 1, 2, 0, 1),  # several row tiles, images ending inside a tile
    (1, 7, 5, 512, 1024, 1, 3, 0, 1),
]


@pytest.mark.parametrize("nb,h,w_,ci,co,k,stride,pad,dil", CONVS)
def test_qconv_parity(K, nb, h, w_, ci, co, k, stride, pad, dil):
    rng = np.random.default_rng(nb * h + ci + co + k)
    x = rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8)
    wt = rng.integers(-128, 128, (co, k, k, ci), dtype=np.int8)
    ho = (h + 2 * pad - dil * (k - 1) - 1) // stride + 1
    wo = (w_ + 2 * pad - dil * (k - 1) - 1) // stride + 1
    md = list(O.NHWC_OHWI_METADATA) + [stride, stride, dil, dil, 1]
    padding = [pad, pad, pad, pad]
    out_shape = [nb, ho, wo, co]
    acc = O.conv_s32(x, wt, padding, md, out_shape)
    names = K.variant_names()
    variants = [-1, 0] + ([i for i, nm in enumerate(names) if nm.startswith(("mfma_", "pipe_", "dual_"))]
                          if ci % 16 == 0 else [])
    if k == 3 and stride == 1 and dil == 1 and ci in (32, 64, 128, 256):
        for i, nm in enumerate(names):
            if not nm.startswith("direct3x3_"):
                continue
            try:      # (a tile whose input patch does not fit the LDS for this shape is refused)
                K.qconv2d(dev(x), dev(wt), padding, md, out_shape, K.EPI_ACC_S32, variant=i)
                variants.append(i)
            except RuntimeError as exc:
                assert "fits the LDS" in str(exc) and nm == "direct3x3_512x64", (nm, exc)
    for v in variants:
        got = host(K.qconv2d(dev(x), dev(wt), padding, md, out_shape, K.EPI_ACC_S32, variant=v))
        np.testing.assert_array_equal(got, acc, err_msg="variant %d" % v)
    sx, sw = make_scales(rng, co)
    so = pick_so(acc, sx, sw)
    want = O.requant_cpu(acc.reshape(-1, co), sx, sw, so).reshape(out_shape)
    for v in variants:
        got = host(K.qconv2d(dev(x), dev(wt), padding, md, out_shape, K.EPI_REQUANT_CPU,
                             sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])), variant=v))
        np.testing.assert_array_equal(got, want, err_msg="variant %d" % v)
    # the integer output stage of the reference's AArch64 convolution, with an s32 bias
    b32 = rng.integers(-100000, 100000, co).astype(np.int32)
    want_fx = O.requant_fixedpoint(acc.reshape(-1, co), sx, sw, so, b32=b32, zo=-2).reshape(out_shape)
    for v in variants:
        got = host(K.qconv2d(dev(x), dev(wt), padding, md, out_shape, K.EPI_REQUANT_FIXEDPOINT,
                             sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])),
                             bias=dev(b32), zo=-2, variant=v))
        np.testing.assert_array_equal(got, want_fx, err_msg="fixed-point, variant %d" % v)
    # requant -> dequantize in the convolution's epilogue: the bits of dequantize(requant)
    want_f = O.dequantize(want, np.array([so], np.float32), np.array([0], np.int32))
    for v in variants:
        got = host(K.qconv2d(dev(x), dev(wt), padding, md, out_shape, K.EPI_REQUANT_CPU_DEQUANT_F32,
                             sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])), variant=v))
        assert got.dtype == np.float32
        assert np.array_equal(got.view(np.uint32), want_f.view(np.uint32)), "variant %d" % v


@pytest.mark.parametrize("nb,h,w_,ci,co,k,pad", [(2, 14, 14, 64, 256, 1, 0), (1, 28, 28, 128, 128, 3, 1),
                                                 (2, 9, 11, 48, 72, 3, 1), (1, 7, 7, 24, 40, 1, 0),
                                                 # the kernel with the input patch resident in LDS
                                                 (64, 32, 32, 32, 32, 3, 1), (32, 56, 56, 64, 64, 3, 1)])
def test_qconv_fused_residual_relu_quantize(K, nb, h, w_, ci, co, k, pad):
    """The tail of a ResNet block in the convolution's epilogue: dequantize -> + the block's
    int8 input (its own scale and zero point) -> ReLU -> quantize gives the bits of the
    separate library calls; so does an f32 residual with an f32 result, and a table."""
    rng = np.random.default_rng(h * 31 + ci + co)
    x = dev(rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8))
    wt = dev(rng.integers(-128, 128, (co, k, k, ci), dtype=np.int8))
    md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
    padding = [pad] * 4
    out_shape = [nb, h, w_, co]
    acc = O.conv_s32(host(x), host(wt), padding, md, out_shape)
    sx, sw = make_scales(rng, co)
    so = pick_so(acc, sx, sw)
    sc = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so], np.float32)))
    bias = dev((rng.standard_normal(co) * 10 * so).astype(np.float32))
    q = K.qconv2d(x, wt, padding, md, out_shape, K.EPI_REQUANT_CPU, bias=bias, zo=2, **sc)
    zi = lambda v: torch.full((1,), v, dtype=torch.int32, device="cuda")  # noqa: E731
    y = K.dequantize(q, sc["so"], zi(2))
    rq = dev(rng.integers(-128, 128, out_shape, dtype=np.int8))
    rs, rz = dev(np.array([so * 0.8], np.float32)), -5
    s2, z2 = dev(np.array([so * 1.1], np.float32)), -128
    t = y + K.dequantize(rq, rs, zi(rz))
    t = torch.where(t < 0, torch.zeros_like(t), t)
    want = K.quantize(t, s2, zi(z2))
    got = K.qconv2d(x, wt, padding, md, out_shape, K.EPI_REQUANT_CPU, bias=bias, zo=2, **sc,
                    post=K.make_postops(residual=rq, residual_scale=rs, residual_zp=rz,
                                        relu=True, out_scale=s2, out_zp=z2))
    assert torch.equal(got, want)
    rf = dev((rng.standard_normal(out_shape) * 40 * so).astype(np.float32))
    got = K.qconv2d(x, wt, padding, md, out_shape, K.EPI_REQUANT_CPU_DEQUANT_F32, bias=bias, zo=2,
                    **sc, post=K.make_postops(residual=rf))
    assert torch.equal(got.view(torch.int32), (y + rf).view(torch.int32))
    table = dev(rng.integers(-128, 128, 256, dtype=np.int8))
    got = K.qconv2d(x, wt, padding, md, out_shape, K.EPI_REQUANT_CPU, bias=bias, zo=2, **sc,
                    post=K.make_postops(table=table))
    assert torch.equal(got, K.lut8(q, table))


def test_qconv_1x1_with_many_tiles_keeps_the_fixed_point_stage_and_fused_operators(K):
    """A 1x1 convolution runs as a plain GEMM over the pixels; with several rounds of tiles the
    plain GEMM would take its persistent kernels, which carry neither the fixed-point stage nor
    fused operators -- the dispatch has to stay on the kernels that do."""
    rng = np.random.default_rng(5)
    nb, h, ci, co = 32, 56, 64, 256                      # 100352 x 64 -> 256: 392 tiles of 256 x 256, two rounds
    x = dev(rng.integers(-128, 128, (nb, h, h, ci), dtype=np.int8))
    wt = dev(rng.integers(-128, 128, (co, 1, 1, ci), dtype=np.int8))
    md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
    osh = [nb, h, h, co]
    acc, _ = O.gemm_s32_fast(host(x).reshape(-1, ci), host(wt).reshape(co, ci))
    sx, sw = make_scales(rng, co)
    so = pick_so(acc, sx, sw)
    sc = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so], np.float32)))
    b32 = rng.integers(-1000, 1000, co).astype(np.int32)
    want = O.requant_fixedpoint(acc, sx, sw, so, b32=b32, zo=1).reshape(osh)
    got = K.qconv2d(x, wt, [0] * 4, md, osh, K.EPI_REQUANT_FIXEDPOINT, bias=dev(b32), zo=1, **sc)
    np.testing.assert_array_equal(host(got), want)
    table = dev(rng.integers(-128, 128, 256, dtype=np.int8))
    q = K.qconv2d(x, wt, [0] * 4, md, osh, K.EPI_REQUANT_CPU, **sc)
    np.testing.assert_array_equal(host(q), O.requant_cpu(acc, sx, sw, so).reshape(osh))
    got = K.qconv2d(x, wt, [0] * 4, md, osh, K.EPI_REQUANT_CPU, **sc, post=K.make_postops(table=table))
    assert torch.equal(got, K.lut8(q, table))
    # the same through the GEMM entry
    a2, w2 = x.reshape(-1, ci), wt.reshape(co, ci)
    got = K.qgemm(a2, w2, K.EPI_REQUANT_FIXEDPOINT, bias=dev(b32), zo=1, **sc)
    np.testing.assert_array_equal(host(got), want.reshape(-1, co))
    got = K.qgemm(a2, w2, K.EPI_REQUANT_CPU, **sc, post=K.make_postops(table=table))
    assert torch.equal(got, K.lut8(q, table).reshape(-1, co))


def test_qconv_direct_random_shapes(K):
    """Seeded sweep for the kernels that keep the input patch in LDS: image sizes that make
    tiles start and end anywhere in a row, every channel count, ragged output channels,
    asymmetric padding, both tile shapes, two epilogues -- bit-exact against the oracle."""
    rng = np.random.default_rng(20250117)
    names = K.variant_names()
    direct = [i for i, nm in enumerate(names) if nm.startswith("direct3x3_")]
    for case in range(24):
        nb = int(rng.integers(1, 4))
        h = int(rng.integers(3, 40))
        w_ = int(rng.integers(3, 70))
        ci = int(rng.choice([32, 64, 128, 256]))
        co = int(rng.choice([8, 17, 64, 72, 130]))
        pad = [int(v) for v in rng.integers(0, 3, 4)]          # top, bottom, left, right
        ho, wo = h + pad[0] + pad[1] - 2, w_ + pad[2] + pad[3] - 2
        if ho < 1 or wo < 1 or (ho + 10) * (wo + 2) * ci > 120 * 1024:
            continue
        x = rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8)
        wt = rng.integers(-128, 128, (co, 3, 3, ci), dtype=np.int8)
        md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
        out_shape = [nb, ho, wo, co]
        acc = O.conv_s32(x, wt, pad, md, out_shape)
        sx, sw = make_scales(rng, co)
        so = pick_so(acc, sx, sw)
        want = O.requant_cpu(acc.reshape(-1, co), sx, sw, so).reshape(out_shape)
        tag = "case %d: %dx%dx%dx%d -> %d pad %s" % (case, nb, h, w_, ci, co, pad)
        for v in direct:
            got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_ACC_S32, variant=v))
            np.testing.assert_array_equal(got, acc, err_msg=tag + " variant %d" % v)
            got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU,
                                 sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])),
                                 variant=v))
            np.testing.assert_array_equal(got, want, err_msg=tag + " variant %d" % v)



def test_qconv_strided_pointwise_rows_are_pixels(K):
    """1 x 1 filters with unequal strides, and with fused operators, on the path that finds each
    GEMM row's input pixel once and then runs the plain GEMM's loop: against the oracle, the
    implicit-GEMM kernel and the separate calls."""
    rng = np.random.default_rng(20260618)
    names = K.variant_names()
    pipe128 = names.index("pipe_128x128x128")
    for nb, h, w_, ci, co, sh, sw_ in [(2, 13, 17, 64, 96, 2, 1), (3, 16, 9, 128, 200, 1, 2), (1, 30, 31, 32, 64, 3, 2),
                                      (16, 28, 28, 256, 512, 2, 2), (4, 56, 56, 64, 128, 2, 2)]:
        x = rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8)
        wt = rng.integers(-128, 128, (co, 1, 1, ci), dtype=np.int8)
        ho, wo = (h - 1) // sh + 1, (w_ - 1) // sw_ + 1
        md = list(O.NHWC_OHWI_METADATA) + [sh, sw_, 1, 1, 1]
        out_shape, pad = [nb, ho, wo, co], [0, 0, 0, 0]
        acc = O.conv_s32(x, wt, pad, md, out_shape)
        tag = "%dx%dx%dx%d -> %d, strides %d %d" % (nb, h, w_, ci, co, sh, sw_)
        np.testing.assert_array_equal(host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_ACC_S32)), acc,
                                      err_msg=tag)
        sx, sw = make_scales(rng, co)
        so = pick_so(acc, sx, sw)
        sc = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])))
        bf = (rng.standard_normal(co) * 30).astype(np.float32)
        got = K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(bf), **sc)
        np.testing.assert_array_equal(host(got), O.requant_gpu(acc.reshape(-1, co), sx, sw, so, bias_f32=bf).reshape(out_shape),
                                      err_msg=tag)
        assert torch.equal(got, K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(bf),
                                          variant=pipe128, **sc)), tag
        plain = K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, **sc)
        res = dev(rng.standard_normal(out_shape).astype(np.float32) * 300)
        s2, z1 = dev(np.array([7.0], np.float32)), torch.zeros(1, dtype=torch.int32, device="cuda")
        fused = K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, **sc,
                          post=K.make_postops(residual=res, relu=True, out_scale=s2, out_zp=-3))
        t = torch.clamp_min(K.dequantize(plain, sc["so"], z1) + res, 0.0)
        assert torch.equal(fused, K.quantize(t, s2, torch.full((1,), -3, dtype=torch.int32, device="cuda"))), tag


def test_qconv_library_choice_on_random_shapes(K):
    """Seeded sweep over what decides the kernel of a convolution -- channel counts with and
    without a register-filter instance, 1 x 1 to 7 x 7 filters, strides, paddings, batch and
    image sizes from one pixel tile to many, ragged output channels, every int8 epilogue and
    bias kind: whatever the library picks gives the bytes of the generic kernel (one thread
    per result; pinned to the oracle by the tests above)."""
    rng = np.random.default_rng(20260507)
    gen = K.variant_names().index("generic")
    md0 = list(O.NHWC_OHWI_METADATA)
    done = 0
    for case in range(500):
        ci = int(rng.choice([3, 4, 16, 32, 64, 64, 128, 128, 256, 256, 512]))
        k = int(rng.choice([7, 3, 5])) if ci <= 4 else int(rng.choice([1, 1, 1, 3, 3, 2]))
        s = int(rng.choice([1, 1, 1, 2]))
        pad = int(rng.choice([0, k // 2, 1 if k > 1 else 0]))
        big = rng.random() < 0.3
        nb = int(rng.integers(1, 40 if big else 6))
        lo, hi = max(k - 2 * pad, 1), 30 if big else 60
        h, w_ = int(rng.integers(lo, hi)), int(rng.integers(lo, hi))
        if ci <= 4:
            h, w_ = 3 * h + 7, 3 * w_ + 7
        co = int(rng.choice([16, 32, 48, 64, 80, 128, 144, 208, 256, 512, 1024, int(rng.integers(1, 300))]))
        ho, wo = (h + 2 * pad - k) // s + 1, (w_ + 2 * pad - k) // s + 1
        if ho < 1 or wo < 1 or nb * ho * wo * co > 3e7 or nb * h * w_ * ci > 3e7:
            continue
        x = dev(rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8))
        wt = dev(rng.integers(-128, 128, (co, k, k, ci), dtype=np.int8))
        out_shape, md = [nb, ho, wo, co], md0 + [s, s, 1, 1, 1]
        so = np.float32(0.02 * 0.025 * 74.0 * 74.0 * np.sqrt(k * k * ci) / 40.0)
        kw = dict(sx=dev(np.array([0.02], np.float32)), sw=dev(rng.uniform(0.001, 0.05, co).astype(np.float32)),
                  so=dev(np.array([so])))
        kind, epi = int(rng.integers(0, 4)), K.EPI_REQUANT_CPU
        if kind == 1:
            kw.update(bias=dev((rng.standard_normal(co) * 3 * so).astype(np.float32)), zo=int(rng.integers(-10, 10)))
        elif kind == 2:
            kw.update(bias=dev(rng.integers(-100000, 100000, co).astype(np.int32)))
        elif kind == 3:
            epi = K.EPI_REQUANT_GPU
            kw.update(bias=dev((rng.standard_normal(co) * 30).astype(np.float32)))
        got = K.qconv2d(x, wt, [pad] * 4, md, out_shape, epi, **kw)
        want = K.qconv2d(x, wt, [pad] * 4, md, out_shape, epi, variant=gen, **kw)
        assert torch.equal(got, want), "case %d: %dx%dx%dx%d, %dx%d stride %d pad %d -> %d, bias kind %d" % (
            case, nb, h, w_, ci, k, k, s, pad, co, kind)
        done += 1
    assert done > 400


def test_qconv_stream_variant(K):
    """The 3 x 3 kernel (64 or 128 input channels) that keeps the filter in registers: images whose pixel
    tiles start and end anywhere in a row, one to many tiles per image, ragged and several
    64-channel slices of output channels, asymmetric padding, both int8 epilogues with every
    bias kind they take and an output zero point -- bit-exact against the oracle; then what it
    must refuse."""
    rng = np.random.default_rng(20260311)
    sv = K.variant_names().index("stream")
    md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
    shapes = [(2, 56, 56, 64, 64, [1, 1, 1, 1]), (1, 3, 3, 64, 16, [1, 1, 1, 1]), (3, 9, 7, 64, 80, [0, 0, 0, 0]),
              (1, 6, 150, 64, 64, [1, 1, 1, 1]), (1, 33, 17, 64, 208, [2, 0, 1, 2]),
              (5, 28, 28, 64, 128, [1, 1, 1, 1]), (1, 112, 112, 64, 64, [1, 1, 1, 1]),
              (40, 14, 14, 64, 64, [0, 2, 2, 0]),
              # 128 input channels: 32-channel slices, several slices per pixel tile
              (3, 28, 28, 128, 128, [1, 1, 1, 1]), (1, 5, 4, 128, 16, [1, 1, 1, 1]),
              (2, 17, 33, 128, 80, [0, 2, 2, 1]), (9, 14, 14, 128, 256, [1, 1, 1, 1]),
              (1, 56, 56, 128, 48, [1, 1, 1, 1])]
    for nb, h, w_, ci, co, pad in shapes:
        ho, wo = h + pad[0] + pad[1] - 2, w_ + pad[2] + pad[3] - 2
        x = rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8)
        wt = rng.integers(-128, 128, (co, 3, 3, ci), dtype=np.int8)
        out_shape = [nb, ho, wo, co]
        acc = O.conv_s32(x, wt, pad, md, out_shape)
        sx, sw = make_scales(rng, co)
        so = pick_so(acc, sx, sw)
        scales = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])))
        tag = "%dx%dx%dx%d -> %d pad %s" % (nb, h, w_, ci, co, pad)
        a2 = acc.reshape(-1, co)
        # E1: plain, f32 bias (folded to s32 as the library does) with an output zero point, s32 bias
        got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, variant=sv, **scales))
        np.testing.assert_array_equal(got, O.requant_cpu(a2, sx, sw, so).reshape(out_shape), err_msg=tag)
        bf = (rng.standard_normal(co) * 40 * so).astype(np.float32)
        b32 = O.bias_f32_to_s32(bf, sx, sw)
        got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, bias=dev(bf), zo=3,
                             variant=sv, **scales))
        np.testing.assert_array_equal(got, O.requant_cpu(a2, sx, sw, so, b32=b32, zo=3).reshape(out_shape),
                                      err_msg=tag + " f32 bias")
        bi = rng.integers(-2000000, 2000000, co).astype(np.int32)
        got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, bias=dev(bi), zo=-5,
                             variant=sv, **scales))
        np.testing.assert_array_equal(got, O.requant_cpu(a2, sx, sw, so, b32=bi, zo=-5).reshape(out_shape),
                                      err_msg=tag + " s32 bias")
        # E2: f32 bias in output units, int8 bias
        bo = (rng.standard_normal(co) * 30).astype(np.float32)
        got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(bo),
                             variant=sv, **scales))
        np.testing.assert_array_equal(got, O.requant_gpu(a2, sx, sw, so, bias_f32=bo).reshape(out_shape),
                                      err_msg=tag + " E2 f32 bias")
        b8 = rng.integers(-128, 128, co, dtype=np.int8)
        got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(b8),
                             variant=sv, **scales))
        np.testing.assert_array_equal(got, O.requant_gpu(a2, sx, sw, so, bias_i8=b8).reshape(out_shape),
                                      err_msg=tag + " E2 s8 bias")
        # the library's own choice for this shape gives the same bytes
        auto = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(b8), **scales))
        np.testing.assert_array_equal(auto, got, err_msg=tag + " heuristic")
    # operators fused behind the convolution run in this kernel too (the library picks it for
    # these shapes): residual (+ ReLU) + quantize and a table, against the separate calls
    for nb, h, w_, ci, co in [(2, 56, 56, 64, 64), (3, 28, 28, 128, 128), (1, 9, 11, 64, 80)]:
        x = dev(rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8))
        wt = dev(rng.integers(-128, 128, (co, 3, 3, ci), dtype=np.int8))
        out_shape = [nb, h, w_, co]
        sc = dict(sx=dev(np.array([0.02], np.float32)), sw=dev(rng.uniform(0.001, 0.05, co).astype(np.float32)),
                  so=dev(np.array([9.0], np.float32)))
        plain = K.qconv2d(x, wt, [1, 1, 1, 1], md, out_shape, K.EPI_REQUANT_CPU, **sc)
        z1 = torch.zeros(1, dtype=torch.int32, device="cuda")
        res = dev(rng.standard_normal(out_shape).astype(np.float32) * 300)
        s2 = dev(np.array([7.0], np.float32))
        for relu in (False, True):
            fused = K.qconv2d(x, wt, [1, 1, 1, 1], md, out_shape, K.EPI_REQUANT_CPU, **sc,
                              post=K.make_postops(residual=res, relu=relu, out_scale=s2, out_zp=-3))
            t = K.dequantize(plain, sc["so"], z1) + res
            if relu:
                t = torch.clamp_min(t, 0.0)
            want = K.quantize(t, s2, torch.full((1,), -3, dtype=torch.int32, device="cuda"))
            assert torch.equal(fused, want), (nb, h, w_, ci, co, relu)
        table = K.activation_table(torch.nn.functional.gelu, sc["so"], z1, s2, z1)
        fused = K.qconv2d(x, wt, [1, 1, 1, 1], md, out_shape, K.EPI_REQUANT_CPU, **sc,
                          post=K.make_postops(table=table))
        assert torch.equal(fused, K.lut8(plain, table))
    # refusals: 4-byte results, other channel counts and filters, strides
    x = dev(rng.integers(-128, 128, (1, 8, 8, 64), dtype=np.int8))
    wt = dev(rng.integers(-128, 128, (64, 3, 3, 64), dtype=np.int8))
    with pytest.raises(RuntimeError, match="streaming variant"):
        K.qconv2d(x, wt, [1, 1, 1, 1], md, [1, 8, 8, 64], K.EPI_ACC_S32, variant=sv)
    one = dev(np.array([0.01], np.float32))
    x32 = dev(rng.integers(-128, 128, (1, 8, 8, 32), dtype=np.int8))
    w32 = dev(rng.integers(-128, 128, (64, 3, 3, 32), dtype=np.int8))
    with pytest.raises(RuntimeError, match="streaming variant"):
        K.qconv2d(x32, w32, [1, 1, 1, 1], md, [1, 8, 8, 64], K.EPI_REQUANT_CPU, sx=one, sw=one, so=one, variant=sv)
    md2 = list(O.NHWC_OHWI_METADATA) + [2, 2, 1, 1, 1]
    with pytest.raises(RuntimeError, match="streaming variant"):
        K.qconv2d(x, wt, [1, 1, 1, 1], md2, [1, 4, 4, 64], K.EPI_REQUANT_CPU, sx=one, sw=one, so=one, variant=sv)


def test_qconv_stream_16_channels(K):
    """4 x 4 filters on 16 channels (what a 7 x 7 stride-2 stem becomes after space to depth) in
    the kernel that keeps the filter in registers: an MFMA step's 32 bytes of k are two
    neighbouring patch pixels.  Bit-exact against the oracle, forced and as the library's choice,
    and the stem itself (3 channels, stride 2) through the library against the oracle."""
    rng = np.random.default_rng(20260413)
    sv = K.variant_names().index("stream")
    md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
    for nb, h, w_, co, pad in [(2, 115, 115, 64, [0, 0, 0, 0]), (1, 9, 12, 80, [1, 2, 0, 3]),
                               (3, 30, 31, 16, [0, 0, 0, 0]), (1, 131, 67, 96, [3, 0, 1, 1]),
                               (9, 20, 20, 64, [0, 0, 0, 0])]:
        ho, wo = h + pad[0] + pad[1] - 3, w_ + pad[2] + pad[3] - 3
        x = rng.integers(-128, 128, (nb, h, w_, 16), dtype=np.int8)
        wt = rng.integers(-128, 128, (co, 4, 4, 16), dtype=np.int8)
        out_shape = [nb, ho, wo, co]
        acc = O.conv_s32(x, wt, pad, md, out_shape)
        sx, sw = make_scales(rng, co)
        so = pick_so(acc, sx, sw)
        scales = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])))
        tag = "%dx%dx%dx16 -> %d pad %s" % (nb, h, w_, co, pad)
        a2 = acc.reshape(-1, co)
        bi = rng.integers(-200000, 200000, co).astype(np.int32)
        got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, bias=dev(bi), zo=-5,
                             variant=sv, **scales))
        np.testing.assert_array_equal(got, O.requant_cpu(a2, sx, sw, so, b32=bi, zo=-5).reshape(out_shape),
                                      err_msg=tag + " s32 bias")
        bo = (rng.standard_normal(co) * 30).astype(np.float32)
        got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(bo),
                             variant=sv, **scales))
        np.testing.assert_array_equal(got, O.requant_gpu(a2, sx, sw, so, bias_f32=bo).reshape(out_shape),
                                      err_msg=tag + " E2 f32 bias")
        auto = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(bo), **scales))
        np.testing.assert_array_equal(auto, got, err_msg=tag + " heuristic")
    # the stem: 7 x 7, stride 2, padding 3, three channels
    md2 = list(O.NHWC_OHWI_METADATA) + [2, 2, 1, 1, 1]
    for nb, h in [(2, 224), (1, 97)]:
        ho = (h + 6 - 7) // 2 + 1
        x = rng.integers(-128, 128, (nb, h, h, 3), dtype=np.int8)
        wt = rng.integers(-128, 128, (64, 7, 7, 3), dtype=np.int8)
        out_shape = [nb, ho, ho, 64]
        acc = O.conv_s32(x, wt, [3, 3, 3, 3], md2, out_shape)
        sx, sw = make_scales(rng, 64)
        so = pick_so(acc, sx, sw)
        got = host(K.qconv2d(dev(x), dev(wt), [3, 3, 3, 3], md2, out_shape, K.EPI_REQUANT_CPU,
                             sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so]))))
        np.testing.assert_array_equal(got, O.requant_cpu(acc.reshape(-1, 64), sx, sw, so).reshape(out_shape),
                                      err_msg="stem %d x %d" % (nb, h))


def test_qconv_stream_pointwise(K):
    """1 x 1 filters on 64 to 256 input channels in the kernel that keeps the filter in registers
    (a GEMM over the pixels with a short k): pixel counts that are and are not a multiple of 16
    (one long row of pixels cut anywhere, or tiles per image), one pixel tile to many, tiles
    that end inside a block of 32 pixels, ragged channel slices, both slice widths of the
    64-channel filter, every bias kind of the int8 epilogues, fused operators -- bit-exact
    against the oracle and against the library's choice; then what it must refuse."""
    rng = np.random.default_rng(20260412)
    names = K.variant_names()
    sv = names.index("stream")
    md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
    pad = [0, 0, 0, 0]
    shapes = [(8, 56, 56, 64, 256), (2, 56, 56, 64, 64), (4, 28, 28, 128, 512), (3, 7, 7, 128, 2048),
              (1, 4, 4, 128, 16), (5, 9, 7, 64, 208), (1, 1, 48, 64, 80), (7, 13, 3, 128, 144),
              (2, 23, 5, 128, 96), (1, 56, 56, 128, 64), (1, 1, 16, 64, 16), (3, 5, 11, 64, 400),
              (1, 1, 33, 64, 48), (16, 112, 112, 64, 64), (1, 300, 301, 128, 128),
              # 256 input channels: 64-channel slices, one round of workgroups and several
              (32, 14, 14, 256, 1024), (3, 9, 7, 256, 208), (2, 56, 56, 256, 64), (1, 5, 3, 256, 16)]
    for nb, h, w_, ci, co in shapes:
        x = rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8)
        wt = rng.integers(-128, 128, (co, 1, 1, ci), dtype=np.int8)
        out_shape = [nb, h, w_, co]
        acc = x.reshape(-1, ci).astype(np.int32) @ wt.reshape(co, ci).astype(np.int32).T
        sx, sw = make_scales(rng, co)
        so = pick_so(acc, sx, sw)
        scales = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])))
        tag = "%dx%dx%dx%d -> %d" % (nb, h, w_, ci, co)
        for v in (sv,):
            got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, variant=v, **scales))
            np.testing.assert_array_equal(got, O.requant_cpu(acc, sx, sw, so).reshape(out_shape), err_msg=tag)
            bf = (rng.standard_normal(co) * 40 * so).astype(np.float32)
            b32 = O.bias_f32_to_s32(bf, sx, sw)
            got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, bias=dev(bf), zo=3,
                                 variant=v, **scales))
            np.testing.assert_array_equal(got, O.requant_cpu(acc, sx, sw, so, b32=b32, zo=3).reshape(out_shape),
                                          err_msg=tag + " f32 bias")
            bi = rng.integers(-2000000, 2000000, co).astype(np.int32)
            got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU, bias=dev(bi), zo=-5,
                                 variant=v, **scales))
            np.testing.assert_array_equal(got, O.requant_cpu(acc, sx, sw, so, b32=bi, zo=-5).reshape(out_shape),
                                          err_msg=tag + " s32 bias")
            bo = (rng.standard_normal(co) * 30).astype(np.float32)
            got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(bo),
                                 variant=v, **scales))
            np.testing.assert_array_equal(got, O.requant_gpu(acc, sx, sw, so, bias_f32=bo).reshape(out_shape),
                                          err_msg=tag + " E2 f32 bias")
            b8 = rng.integers(-128, 128, co, dtype=np.int8)
            got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(b8),
                                 variant=v, **scales))
            np.testing.assert_array_equal(got, O.requant_gpu(acc, sx, sw, so, bias_i8=b8).reshape(out_shape),
                                          err_msg=tag + " E2 s8 bias")
            auto = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_GPU, bias=dev(b8), **scales))
            np.testing.assert_array_equal(auto, got, err_msg=tag + " heuristic")
    # fused operators: residual (+ ReLU) + quantize and a table, against the separate calls
    for nb, h, w_, ci, co in [(32, 28, 28, 64, 256), (2, 28, 28, 128, 512), (1, 9, 11, 64, 80), (40, 56, 56, 128, 128),
                              (8, 14, 14, 256, 1024)]:   # fused on 256 channels: the GEMM tiles' result
        x = dev(rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8))
        wt = dev(rng.integers(-128, 128, (co, 1, 1, ci), dtype=np.int8))
        out_shape = [nb, h, w_, co]
        sc = dict(sx=dev(np.array([0.02], np.float32)), sw=dev(rng.uniform(0.001, 0.05, co).astype(np.float32)),
                  so=dev(np.array([4.0], np.float32)))
        z1 = torch.zeros(1, dtype=torch.int32, device="cuda")
        res = dev(rng.standard_normal(out_shape).astype(np.float32) * 300)
        s2 = dev(np.array([7.0], np.float32))
        plain = K.qconv2d(x, wt, pad, md, out_shape, K.EPI_REQUANT_CPU, variant=sv, **sc)
        for relu in (False, True):
            fused = K.qconv2d(x, wt, pad, md, out_shape, K.EPI_REQUANT_CPU, **sc,
                              post=K.make_postops(residual=res, relu=relu, out_scale=s2, out_zp=-3))
            t = K.dequantize(plain, sc["so"], z1) + res
            if relu:
                t = torch.clamp_min(t, 0.0)
            want = K.quantize(t, s2, torch.full((1,), -3, dtype=torch.int32, device="cuda"))
            assert torch.equal(fused, want), (nb, h, w_, ci, co, relu)
        table = K.activation_table(torch.nn.functional.gelu, sc["so"], z1, s2, z1)
        fused = K.qconv2d(x, wt, pad, md, out_shape, K.EPI_REQUANT_CPU, **sc,
                          post=K.make_postops(table=table))
        assert torch.equal(fused, K.lut8(plain, table)), (nb, h, w_, ci, co)
    # refusals: channel counts without an instance, strides, 4-byte results
    one = dev(np.array([0.01], np.float32))
    for ci, v in ((32, sv), (512, sv)):
        x = dev(rng.integers(-128, 128, (1, 8, 8, ci), dtype=np.int8))
        wt = dev(rng.integers(-128, 128, (64, 1, 1, ci), dtype=np.int8))
        with pytest.raises(RuntimeError, match="streaming variant"):
            K.qconv2d(x, wt, pad, md, [1, 8, 8, 64], K.EPI_REQUANT_CPU, sx=one, sw=one, so=one, variant=v)
    x = dev(rng.integers(-128, 128, (1, 8, 8, 64), dtype=np.int8))
    wt = dev(rng.integers(-128, 128, (64, 1, 1, 64), dtype=np.int8))
    with pytest.raises(RuntimeError, match="streaming variant"):
        K.qconv2d(x, wt, pad, md, [1, 8, 8, 64], K.EPI_ACC_S32, variant=sv)
    md2 = list(O.NHWC_OHWI_METADATA) + [2, 2, 1, 1, 1]
    with pytest.raises(RuntimeError, match="streaming variant"):
        K.qconv2d(x, wt, pad, md2, [1, 4, 4, 64], K.EPI_REQUANT_CPU, sx=one, sw=one, so=one, variant=sv)


def test_qconv_direct_other_filter_sizes(K):
    """The same kernels on filters other than 3 x 3 (up to 7 x 7, rectangular ones too) and on
    16 channels with an even filter width, where an MFMA step's 32 bytes of k are two
    neighbouring patch pixels (the stride-1 form of a stem convolution after space to depth):
    bit-exact against the oracle for every tile shape that accepts the problem."""
    rng = np.random.default_rng(20260303)
    names = K.variant_names()
    direct = [i for i, nm in enumerate(names) if nm.startswith("direct3x3_")]
    ran = 0
    for (nb, h, w_, ci, co, kh, kw, pad) in [
            (2, 20, 30, 32, 64, 5, 5, [2, 2, 2, 2]), (1, 16, 16, 64, 40, 7, 7, [3, 3, 3, 3]),
            (2, 12, 25, 32, 64, 1, 3, [0, 0, 1, 1]), (1, 18, 18, 128, 17, 2, 2, [0, 1, 0, 1]),
            (2, 35, 35, 16, 64, 4, 4, [0, 0, 0, 0]), (3, 19, 40, 16, 48, 2, 2, [1, 0, 0, 1]),
            (1, 60, 115, 16, 64, 4, 4, [0, 0, 0, 0]), (1, 14, 14, 16, 8, 3, 6, [1, 1, 2, 3])]:
        ho, wo = h + pad[0] + pad[1] - kh + 1, w_ + pad[2] + pad[3] - kw + 1
        x = rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8)
        wt = rng.integers(-128, 128, (co, kh, kw, ci), dtype=np.int8)
        md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
        out_shape = [nb, ho, wo, co]
        acc = O.conv_s32(x, wt, pad, md, out_shape)
        sx, sw = make_scales(rng, co)
        so = pick_so(acc, sx, sw)
        want = O.requant_cpu(acc.reshape(-1, co), sx, sw, so).reshape(out_shape)
        tag = "%dx%dx%dx%d -> %d, %dx%d pad %s" % (nb, h, w_, ci, co, kh, kw, pad)
        for v in direct:
            try:
                got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_ACC_S32, variant=v))
            except RuntimeError as exc:
                assert "fits the LDS" in str(exc), (tag, names[v], exc)
                continue
            ran += 1
            np.testing.assert_array_equal(got, acc, err_msg=tag + " " + names[v])
            got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_REQUANT_CPU,
                                 sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])),
                                 variant=v))
            np.testing.assert_array_equal(got, want, err_msg=tag + " " + names[v])
        got = host(K.qconv2d(dev(x), dev(wt), pad, md, out_shape, K.EPI_ACC_S32))
        np.testing.assert_array_equal(got, acc, err_msg=tag + " auto")
    assert ran >= 20
    # 16 channels and an odd filter width: no layout for that
    x = rng.integers(-128, 128, (1, 8, 8, 16), dtype=np.int8)
    wt = rng.integers(-128, 128, (8, 3, 3, 16), dtype=np.int8)
    md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
    for v in direct:
        with pytest.raises(RuntimeError, match="direct variants"):
            K.qconv2d(dev(x), dev(wt), [1] * 4, md, [1, 8, 8, 8], K.EPI_ACC_S32, variant=v)


def test_qconv_direct_variants_refuse_what_they_cannot_run(K):
    """A named direct-convolution variant fails with an error, not a wrong result, on a
    filter of a single tap or a stride other than 1, on a channel count it has no layout for, and on an image
    row too wide for its patch to fit the LDS; the automatic choice runs all of them."""
    names = K.variant_names()
    direct = [i for i, nm in enumerate(names) if nm.startswith("direct3x3_")]
    assert direct
    rng = np.random.default_rng(5)
    cases = [  # nb, h, w, ci, co, k, stride
        (1, 8, 8, 64, 64, 1, 1),
        (1, 9, 9, 64, 64, 3, 2),
        (1, 8, 8, 48, 64, 3, 1),
        (1, 4, 300, 256, 64, 3, 1),
    ]
    for nb, h, w_, ci, co, k, stride in cases:
        pad = k // 2
        x = rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8)
        wt = rng.integers(-128, 128, (co, k, k, ci), dtype=np.int8)
        ho = (h + 2 * pad - k) // stride + 1
        wo = (w_ + 2 * pad - k) // stride + 1
        md = list(O.NHWC_OHWI_METADATA) + [stride, stride, 1, 1, 1]
        out_shape = [nb, ho, wo, co]
        for v in direct:
            with pytest.raises(RuntimeError, match="direct variants"):
                K.qconv2d(dev(x), dev(wt), [pad] * 4, md, out_shape, K.EPI_ACC_S32, variant=v)
        got = host(K.qconv2d(dev(x), dev(wt), [pad] * 4, md, out_shape, K.EPI_ACC_S32))
        np.testing.assert_array_equal(got, O.conv_s32(x, wt, [pad] * 4, md, out_shape))


def test_qconv_nchw_oihw_generic(K):
    rng = np.random.default_rng(77)
    x = rng.integers(-128, 128, (2, 4, 6, 6), dtype=np.int8)       # NCHW
    wt = rng.integers(-128, 128, (3, 4, 3, 3), dtype=np.int8)      # OIHW
    md = [0, 1, 2, 3, 1, 0, 2, 3, 0, 1, 2, 3, 1, 1, 1, 1, 1]
    acc = O.conv_s32(x, wt, [1, 1, 1, 1], md, [2, 3, 6, 6])
    got = host(K.qconv2d(dev(x), dev(wt), [1, 1, 1, 1], md, [2, 3, 6, 6], K.EPI_ACC_S32))
    np.testing.assert_array_equal(got, acc)


@pytest.mark.parametrize("nb,ci,h,w_,co,k,stride,pad,dil", [(2, 32, 14, 14, 48, 3, 1, 1, 1), (3, 24, 9, 11, 40, 3, 2, 1, 1),
                                                         (1, 64, 28, 28, 64, 1, 1, 0, 1), (2, 16, 12, 12, 20, 3, 1, 2, 2)])
def test_qconv_nchw_oihw_on_the_mfma_path(K, nb, ci, h, w_, co, k, stride, pad, dil):
    """NCHW x OIHW -> NCHW with scratch: tensors re-laid out as NHWC / OHWI, MFMA kernels, result
    turned back -- the same bits as the oracle and as the generic kernel without scratch, for
    every epilogue family (int8, int32 and f32 results)."""
    rng = np.random.default_rng(ci + co + h)
    x = rng.integers(-128, 128, (nb, ci, h, w_), dtype=np.int8)
    wt = rng.integers(-128, 128, (co, ci, k, k), dtype=np.int8)
    ho = (h + 2 * pad - dil * (k - 1) - 1) // stride + 1
    wo = (w_ + 2 * pad - dil * (k - 1) - 1) // stride + 1
    md = [0, 1, 2, 3, 1, 0, 2, 3, 0, 1, 2, 3, stride, stride, dil, dil, 1]
    padding, osh = [pad] * 4, [nb, co, ho, wo]
    acc = O.conv_s32(x, wt, padding, md, osh)
    for ws in (True, False):
        got = host(K.qconv2d(dev(x), dev(wt), padding, md, osh, K.EPI_ACC_S32, workspace=ws))
        np.testing.assert_array_equal(got, acc)
    sx, sw = make_scales(rng, co)
    so = pick_so(acc, sx, sw)
    sc = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so], np.float32)))
    per_c = lambda a: np.moveaxis(a, 1, -1).reshape(-1, co)                      # noqa: E731
    back = lambda a: np.moveaxis(a.reshape(nb, ho, wo, co), -1, 1)               # noqa: E731
    want = back(O.requant_cpu(per_c(acc), sx, sw, so))
    got = host(K.qconv2d(dev(x), dev(wt), padding, md, osh, K.EPI_REQUANT_CPU, **sc))
    np.testing.assert_array_equal(got, want)
    b32 = rng.integers(-100000, 100000, co).astype(np.int32)
    want = back(O.requant_fixedpoint(per_c(acc), sx, sw, so, b32=b32, zo=3))
    got = host(K.qconv2d(dev(x), dev(wt), padding, md, osh, K.EPI_REQUANT_FIXEDPOINT, bias=dev(b32),
                         zo=3, **sc))
    np.testing.assert_array_equal(got, want)
    got_f = host(K.qconv2d(dev(x), dev(wt), padding, md, osh, K.EPI_REQUANT_CPU_DEQUANT_F32, **sc))
    want_f = O.dequantize(back(O.requant_cpu(per_c(acc), sx, sw, so)), np.array([so], np.float32),
                          np.array([0], np.int32))
    assert np.array_equal(got_f.view(np.uint32), want_f.view(np.uint32))


@pytest.mark.parametrize("nb,ci,h,w_,co,k,pads", [(2, 3, 32, 32, 64, 7, (3, 3, 3, 3)), (1, 3, 17, 23, 20, 7, (3, 2, 2, 3)),
                                                 (3, 1, 12, 12, 16, 3, (1, 1, 1, 1)), (2, 4, 15, 14, 33, 5, (2, 2, 2, 2)),
                                                 (1, 2, 9, 9, 8, 2, (0, 0, 0, 0)), (2, 3, 8, 8, 64, 3, (0, 1, 0, 1)),
                                                 (1, 3, 4, 4, 8, 7, (3, 3, 3, 3))])
def test_qconv_stride2_few_channels_space_to_depth(K, nb, ci, h, w_, co, k, pads):
    """Stride-2 convolutions of images with at most 4 channels (the 7 x 7 stem of a vision
    network): with scratch they run as a stride-1 convolution of the space-to-depth image on
    the MFMA kernels -- the same bits as the oracle and as the path without scratch; odd and
    even filter sizes, asymmetric padding, odd image sizes, an image so small that the
    space-to-depth copy is larger than the padded one, NCHW x OIHW on top."""
    rng = np.random.default_rng(ci * 100 + k + h)
    x = rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8)
    wt = rng.integers(-128, 128, (co, k, k, ci), dtype=np.int8)
    ho = (h + pads[0] + pads[1] - k) // 2 + 1
    wo = (w_ + pads[2] + pads[3] - k) // 2 + 1
    md = list(O.NHWC_OHWI_METADATA) + [2, 2, 1, 1, 1]
    padding, osh = list(pads), [nb, ho, wo, co]
    acc = O.conv_s32(x, wt, padding, md, osh)
    for ws in (True, False):
        got = host(K.qconv2d(dev(x), dev(wt), padding, md, osh, K.EPI_ACC_S32, workspace=ws))
        np.testing.assert_array_equal(got, acc)
    sx, sw = make_scales(rng, co)
    so = pick_so(acc, sx, sw)
    sc = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so], np.float32)))
    want = O.requant_cpu(acc.reshape(-1, co), sx, sw, so).reshape(osh)
    got = host(K.qconv2d(dev(x), dev(wt), padding, md, osh, K.EPI_REQUANT_CPU, **sc))
    np.testing.assert_array_equal(got, want)
    # the PyTorch layouts: NCHW x OIHW -> NCHW
    md_t = [0, 1, 2, 3, 1, 0, 2, 3, 0, 1, 2, 3, 2, 2, 1, 1, 1]
    x_t, w_t = np.ascontiguousarray(np.moveaxis(x, -1, 1)), np.ascontiguousarray(np.moveaxis(wt, -1, 1))
    got = host(K.qconv2d(dev(x_t), dev(w_t), padding, md_t, [nb, co, ho, wo], K.EPI_REQUANT_CPU, **sc))
    np.testing.assert_array_equal(got, np.moveaxis(want, -1, 1))


def test_qconv_known_answers(K, golden):
    for case in golden["qconv"]:
        if case["data_format"] != "NHWC":
            continue
        x = np.full(case["in_shape"], case["x"], np.float32)
        w = np.full(case["w_hwio"], case["w"], np.float32)
        co = w.shape[3]
        sw = np.full(co, case["sw"], np.float32)
        qx = O.quantize(x, case["sx"], 0)
        qw = np.ascontiguousarray(O.quantize(w, sw, np.zeros(co, np.int32), axis=3).transpose(3, 0, 1, 2))
        pad, md, out_shape = O.conv_attrs(qx.shape, qw.shape, "NHWC", case["strides"],
                                          case["dilations"], case["padding"])
        out = host(K.qconv2d(dev(qx), dev(qw), pad, md, out_shape, K.EPI_REQUANT_CPU,
                             sx=dev(np.array([case["sx"]], np.float32)), sw=dev(sw),
                             so=dev(np.array([case["so"]], np.float32))))
        if case["padding"] == "VALID" or case["w_hwio"][0] == 1 or case["x"] == 0.0:
            assert (out.astype(np.float32) * case["so"] == case["expect_f32"]).all(), case["src"]


@pytest.mark.parametrize("m,n,k,pad", [(300, 200, 256, 64), (17, 48, 1040, 16), (1000, 768, 768, 128)])
def test_qgemm_strided_rows_all_variants(K, m, n, k, pad):
    """Operands and output that are column slices of wider buffers (row stride > row
    length): the kernels must neither read the gap as data nor write into it."""
    rng = np.random.default_rng(m + n + k)
    a_full = rng.integers(-128, 128, (m, k + pad), dtype=np.int8)
    w_full = rng.integers(-128, 128, (n, k + 2 * pad), dtype=np.int8)
    a, w = a_full[:, :k], w_full[:, pad:pad + k]
    acc, _ = O.gemm_s32_fast(np.ascontiguousarray(a), np.ascontiguousarray(w))
    sx, sw = make_scales(rng, n)
    so = pick_so(acc, sx, sw)
    want = O.requant_cpu(acc, sx, sw, so)
    da, dw = dev(a_full)[:, :k], dev(w_full)[:, pad:pad + k]
    for v in [-1] + gemm_variants(K, k, n + pad):
        out_full = torch.full((m, n + pad), 77, dtype=torch.int8, device="cuda")
        K.qgemm(da, dw, K.EPI_REQUANT_CPU, sx=dev(np.array([sx])), sw=dev(sw),
                so=dev(np.array([so])), out=out_full[:, :n], variant=v)
        got = host(out_full)
        np.testing.assert_array_equal(got[:, :n], want, err_msg="variant %d" % v)
        assert (got[:, n:] == 77).all(), "variant %d wrote past the row" % v


@pytest.mark.parametrize("m,n,k", [(70, 33, 64), (300, 129, 256), (500, 1501, 80), (2100, 515, 128), (4200, 1027, 64)])
def test_qgemm_4_byte_results_in_rows_at_any_word(K, m, n, k):
    """int32 and f32 results in rows that begin at any multiple of four bytes, also with a residual at
    another one: 16 bytes a lane, the row's end element by element, nothing beside the rows."""
    rng = np.random.default_rng(m + n + k)
    a, w = dev(rng.integers(-128, 128, (m, k), dtype=np.int8)), dev(rng.integers(-128, 128, (n, k), dtype=np.int8))
    sw = dev(rng.uniform(0.001, 0.05, n).astype(np.float32))
    sc = dict(sx=dev(np.array([0.02], np.float32)), sw=sw, so=dev(np.array([0.3], np.float32)))
    bias = dev(rng.standard_normal(n).astype(np.float32))
    wide = torch.zeros((m, n + 3), device="cuda")
    res = wide[:, 2:n + 2]
    res.copy_(dev(rng.standard_normal((m, n)).astype(np.float32)))
    for epi, kw in ((K.EPI_ACC_S32, {}), (K.EPI_DEQUANT_F32, dict(sx=sc["sx"], sw=sw, bias=bias)),
                    (K.EPI_REQUANT_CPU_DEQUANT_F32, dict(bias=bias, **sc))):
        want = K.qgemm(a, w, epi, variant=0, **kw).view(torch.int32)
        for lead in range(4):
            frame = torch.full((m, n + 4), 77, dtype=torch.int32, device="cuda")
            out = frame if epi == K.EPI_ACC_S32 else frame.view(torch.float32)
            K.qgemm(a, w, epi, out=out[:, lead:lead + n], **kw)
            assert torch.equal(frame[:, lead:lead + n], want), (epi, lead)
            assert bool((frame[:, :lead] == 77).all()) and bool((frame[:, lead + n:] == 77).all()), (epi, lead)
    y = K.qgemm(a, w, epi, variant=0, **kw)
    got = K.qgemm(a, w, epi, post=K.make_postops(residual=res), **kw)
    assert torch.equal(got.view(torch.int32), (y + res).view(torch.int32))


@pytest.mark.parametrize("m,n,k,ldo", [(300, 200, 256, 208), (1000, 100, 768, 112), (513, 72, 128, 80),
                                       (4100, 1000, 768, 1008), (260, 328, 512, 336)])
def test_qgemm_ragged_channels_in_16_byte_aligned_rows(K, m, n, k, ldo):
    """Output rows that take 16-byte stores (aligned buffer, row stride a multiple of 16) while
    the channel count is not a multiple of 16: the last chunk of a row is written byte by byte,
    and nothing lands in the columns behind it -- every variant, both int8 epilogues."""
    rng = np.random.default_rng(m * 7 + n)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc, _ = O.gemm_s32_fast(a, w)
    sx, sw = make_scales(rng, n)
    so = pick_so(acc, sx, sw)
    bias = rng.standard_normal(n).astype(np.float32) * 5
    want1 = O.requant_cpu(acc, sx, sw, so)
    want2 = O.requant_gpu(acc, sx, sw, so, bias_f32=bias)
    da, dw = dev(a), dev(w)
    scales = dict(sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])))
    for v in [-1] + gemm_variants(K, k, ldo):
        for epi, want, b in ((K.EPI_REQUANT_CPU, want1, None), (K.EPI_REQUANT_GPU, want2, dev(bias))):
            out_full = torch.full((m, ldo), 77, dtype=torch.int8, device="cuda")
            K.qgemm(da, dw, epi, bias=b, out=out_full[:, :n], variant=v, **scales)
            got = host(out_full)
            np.testing.assert_array_equal(got[:, :n], want, err_msg="variant %d epilogue %d" % (v, epi))
            assert (got[:, n:] == 77).all(), "variant %d wrote past the row" % v


def test_qgemm_random_shapes_epilogues_variants(K):
    """Seeded sweep over ragged shapes, every epilogue / bias kind and every kernel
    variant (heuristic included), bit-exact against the oracle."""
    rng = np.random.default_rng(20240611)
    choices = [-1] + gemm_variants(K, 16)
    for case in range(80):
        m = int(rng.choice([1, 2, 7, 16, 31, 33, 64, 100, 129, 255, 300, 513, 1000]))
        n = int(rng.choice([1, 3, 16, 17, 48, 64, 65, 130, 256, 300, 768]))
        k = int(rng.choice([16, 32, 48, 64, 112, 128, 144, 256, 400, 768, 1040]))
        a = rng.integers(-128, 128, (m, k), dtype=np.int8)
        w = rng.integers(-128, 128, (n, k), dtype=np.int8)
        acc, _ = O.gemm_s32_fast(a, w)
        sx, sw = make_scales(rng, n, per_channel=bool(rng.integers(0, 2)))
        so = pick_so(acc, sx, np.broadcast_to(sw, (n,)))
        v = choices[int(rng.integers(0, len(choices)))]
        epi = int(rng.integers(0, 4))
        if persistent_refuses(K, v, n, 4 if epi in (0, 3) else 1):
            v = -1
        tag = "case %d: %dx%dx%d variant %d epilogue %d" % (case, m, n, k, v, epi)
        da, dw = dev(a), dev(w)
        dsx, dsw, dso = dev(np.array([sx])), dev(sw), dev(np.array([so]))
        if epi == 0:
            got = host(K.qgemm(da, dw, K.EPI_ACC_S32, variant=v))
            np.testing.assert_array_equal(got, acc, err_msg=tag)
        elif epi == 1:
            kind = int(rng.integers(0, 3))
            bias = [None, rng.integers(-5000, 5000, n).astype(np.int32),
                    rng.standard_normal(n).astype(np.float32)][kind]
            b32 = bias if kind != 2 else O.bias_f32_to_s32(bias, float(sx), np.broadcast_to(sw, (n,)))
            zo = int(rng.integers(-5, 6))
            want = O.requant_cpu(acc, float(sx), sw, float(so), b32=b32, zo=zo)
            got = host(K.qgemm(da, dw, K.EPI_REQUANT_CPU, sx=dsx, sw=dsw, so=dso,
                               bias=None if bias is None else dev(bias), zo=zo, variant=v))
            np.testing.assert_array_equal(got, want, err_msg=tag)
        elif epi == 2:
            kind = int(rng.integers(0, 3))
            bias = [None, rng.standard_normal(n).astype(np.float32) * 5,
                    rng.integers(-128, 128, n, dtype=np.int8)][kind]
            want = O.requant_gpu(acc, sx, sw, so, bias_f32=bias if kind == 1 else None,
                                 bias_i8=bias if kind == 2 else None)
            got = host(K.qgemm(da, dw, K.EPI_REQUANT_GPU, sx=dsx, sw=dsw, so=dso,
                               bias=None if bias is None else dev(bias), variant=v))
            np.testing.assert_array_equal(got, want, err_msg=tag)
        else:
            bias = rng.standard_normal(n).astype(np.float32) if rng.integers(0, 2) else None
            want = O.dequant_acc(acc, float(sx), sw, bias=bias)
            got = host(K.qgemm(da, dw, K.EPI_DEQUANT_F32, sx=dsx, sw=dsw,
                               bias=None if bias is None else dev(bias), variant=v))
            np.testing.assert_array_equal(got, want, err_msg=tag)


def test_requant_nan_and_inf_scales_saturate_like_the_oracle(K):
    """A NaN or infinite per-channel factor: NaN results go to -128, infinities
    saturate by sign, on every kernel family and both requant epilogues."""
    rng = np.random.default_rng(11)
    m, n, k = 130, 256, 256
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    acc, _ = O.gemm_s32_fast(a, w)
    sx = np.float32(0.02)
    sw = rng.uniform(0.001, 0.05, n).astype(np.float32)
    sw[3] = np.nan
    sw[7] = np.inf
    sw[200] = -np.inf
    so = np.float32(2.0)
    bias = rng.standard_normal(n).astype(np.float32)
    with np.errstate(all="ignore"):
        want_gpu = O.requant_gpu(acc, sx, sw, so, bias_f32=bias)
        want_cpu = O.requant_cpu(acc, sx, sw, so)
    assert (want_gpu[:, 3] == -128).all()
    for v in gemm_variants(K, k, n):
        got = host(K.qgemm(dev(a), dev(w), K.EPI_REQUANT_GPU, sx=dev(np.array([sx])), sw=dev(sw),
                           so=dev(np.array([so])), bias=dev(bias), variant=v))
        np.testing.assert_array_equal(got, want_gpu, err_msg="variant %d" % v)
        got = host(K.qgemm(dev(a), dev(w), K.EPI_REQUANT_CPU, sx=dev(np.array([sx])), sw=dev(sw),
                           so=dev(np.array([so])), variant=v))
        np.testing.assert_array_equal(got, want_cpu, err_msg="variant %d" % v)


def test_bad_arguments_fail_loudly(K):
    a = torch.zeros((4, 16), dtype=torch.int8, device="cuda")
    w = torch.zeros((4, 32), dtype=torch.int8, device="cuda")
    with pytest.raises(ValueError):
        K.qgemm(a, w, K.EPI_ACC_S32)
    w = torch.zeros((4, 16), dtype=torch.int8, device="cuda")
    with pytest.raises(RuntimeError):
        K.qgemm(a, w, K.EPI_REQUANT_CPU)          # scales missing
    with pytest.raises(RuntimeError):
        K.qgemm(a, w, K.EPI_ACC_S32, variant=99)
    # limits are checked before any pointer is touched
    from bladedisc_amd import _lib
    L = _lib.lib()
    import ctypes as C
    big = C.c_int64(1 << 31)
    one = C.c_int64(1)
    st = L.dq8_qgemm(None, one, None, one, None, big, one, big, one, 0, 1, 0, None, 0, None, one,
                     None, one, None, one, 0, 0, 0, None, C.c_size_t(0), None)
    assert st != 0 and b"2^31" in L.dq8_last_error()
    st = L.dq8_qgemm(None, one, None, one, None, one, C.c_int64(-1), one, one, 0, 1, 0, None, 0,
                     None, one, None, one, None, one, 0, 0, 0, None, C.c_size_t(0), None)
    assert st != 0 and b"negative" in L.dq8_last_error()


@pytest.mark.parametrize("m,k,n", [(64, 768, 768), (1, 768, 768), (16, 768, 3072), (33, 3072, 768),
                                   (128, 768, 768), (7, 80, 24), (50, 1024, 200), (32, 768, 2304)])
@pytest.mark.parametrize("epi_name", ["REQUANT_CPU", "REQUANT_GPU", "REQUANT_CPU_DEQUANT_F32",
                                      "DEQUANT_F32", "ACC_S32"])
def test_qlinear_f32_equals_quantize_then_qgemm(K, m, k, n, epi_name):
    """The one-launch quantized linear on f32 activations against the oracle's quantize ->
    gemm -> epilogue and against the library's own two operators: the same bits.  Activations
    include exact rounding ties (multiples of scale / 2), values beyond the int8 range, zeros,
    and infinities; both rounding modes.  (A NaN activation is compared between the two forms of
    the library only: the reference leaves its quantized value undefined.)"""
    rng = np.random.default_rng(m + k + n)
    sx = np.float32(rng.uniform(0.01, 0.05))
    x = rng.standard_normal((m, k)).astype(np.float32)
    ties = rng.integers(-300, 300, x.shape).astype(np.float32) * np.float32(0.5) * sx
    x = np.where(rng.random(x.shape) < 0.1, ties, x).astype(np.float32)
    x.flat[0] = 0.0
    if x.size > 8:
        x.flat[3], x.flat[4] = np.inf, -np.inf
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    sw = rng.uniform(0.001, 0.05, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    epi = getattr(K, "EPI_" + epi_name)
    for round_mode in (K.ROUND_HALF_TO_EVEN, K.ROUND_HALF_AWAY_FROM_ZERO):
        xq = O.quantize(x, sx, 0, round_mode=round_mode)
        acc = O.gemm_s32(xq, w, tp_b=True)
        so = pick_so(acc, sx, sw)
        b = None if epi_name == "ACC_S32" else bias
        got = K.qlinear_f32(dev(x), dev(w), epi, dev(np.array([sx])), dev(sw), dev(np.array([so])),
                            bias=dev(b) if b is not None else None, round_mode=round_mode)
        dxq = K.quantize(dev(x), dev(np.array([sx])), dev(np.zeros(1, np.int32)), round_mode=round_mode)
        np.testing.assert_array_equal(host(dxq), xq)
        two = K.qgemm(dxq, dev(w), epi, sx=dev(np.array([sx])), sw=dev(sw), so=dev(np.array([so])),
                      bias=dev(b) if b is not None else None)
        np.testing.assert_array_equal(host(got).view(np.uint8), host(two).view(np.uint8))
        if x.size > 8:
            xn = x.copy()
            xn.flat[6] = np.nan
            args = (dev(w), epi, dev(np.array([sx])), dev(sw), dev(np.array([so])))
            got_n = K.qlinear_f32(dev(xn), *args, bias=dev(b) if b is not None else None,
                                  round_mode=round_mode)
            xnq = K.quantize(dev(xn), dev(np.array([sx])), dev(np.zeros(1, np.int32)), round_mode=round_mode)
            two_n = K.qgemm(xnq, dev(w), epi, sx=args[2], sw=args[3], so=args[4],
                            bias=dev(b) if b is not None else None)
            np.testing.assert_array_equal(host(got_n).view(np.uint8), host(two_n).view(np.uint8))
        if epi_name == "REQUANT_CPU":
            want = O.requant_cpu(acc, sx, sw, so, b32=O.bias_f32_to_s32(bias, sx, sw))
        elif epi_name == "REQUANT_GPU":
            want = O.requant_gpu(acc, sx, sw, so, bias_f32=bias)
        elif epi_name == "ACC_S32":
            want = acc
        else:
            continue
        np.testing.assert_array_equal(host(got), want)


def test_qlinear_f32_refuses_more_rows_than_it_pays_for(K):
    n, k = 768, 768
    rows = K.qlinear_f32_fused_max_rows(n, k)
    assert 64 <= rows <= 4096 and K.qlinear_f32_fused_max_rows(n, 100) == 0
    x = torch.zeros((rows + 1, k), device="cuda")
    w = torch.zeros((n, k), dtype=torch.int8, device="cuda")
    one = torch.ones(1, device="cuda")
    with pytest.raises(RuntimeError, match="fused_max_rows"):
        K.qlinear_f32(x, w, K.EPI_ACC_S32, one)


def _weight_only_case(rng, m, k, n, dtype, signed):
    npdt = np.float16 if dtype == torch.float16 else np.float32
    x = rng.standard_normal((m, k)).astype(npdt)
    if signed:
        w = rng.integers(-128, 128, (n, k), dtype=np.int8)
        zp = rng.integers(-8, 9, n).astype(np.int32)
    else:
        w = rng.integers(0, 256, (n, k), dtype=np.uint8)
        zp = rng.integers(118, 139, n).astype(np.int32)
    scale = rng.uniform(0.002, 0.02, n).astype(npdt)
    bias = rng.standard_normal(n).astype(npdt)
    return x, w, scale, zp, bias


def _weight_only_plan(m, n, k, dtype, ragged=False):
    """(tile form, k ranges) of a weight-only product that has all the scratch it wants."""
    import ctypes as C
    import bladedisc_amd._lib as _lib
    plan = (C.c_int * 4)()
    _lib.hooks().dq8_weight_only_plan(m, n, k, 1 if dtype == torch.float16 else 0, int(ragged), plan)
    return plan[0], plan[1]


def _weight_only_raw(x, w, scale, zp, bias, out, ws, ws_bytes):
    """The C entry on device matrices whose rows may be pieces of wider ones, the weights' too (which
    kernels.weight_only_qgemm makes contiguous first)."""
    import bladedisc_amd._lib as _lib
    L = _lib.lib()
    (m, k), n = x.shape, w.shape[0]
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    _lib.check(L.dq8_weight_only_qgemm(
        ptr(x), 1 if x.dtype == torch.float16 else 0, x.stride(0), ptr(w), int(w.dtype == torch.int8), w.stride(0), 1,
        ptr(scale), ptr(zp), ptr(bias), ptr(out), out.stride(0), m, n, k, ptr(ws), ws_bytes,
        torch.cuda.current_stream().cuda_stream), "dq8_weight_only_qgemm")


def _weight_only_framed(x, w, dtype, signed):
    """Device copies of both operands inside wider buffers of NaN / the largest byte."""
    (m, k), n = x.shape, w.shape[0]
    wide_x = torch.full((m + 1, k + 16), float("nan"), dtype=dtype, device="cuda")
    wide_x[:m, :k] = dev(x)
    wide_w = torch.full((n + 1, k + 16), -1 if signed else 255, dtype=torch.int8 if signed else torch.uint8,
                        device="cuda")
    wide_w[:n, :k] = dev(w)
    return wide_x[:m, :k], wide_w[:n, :k]


def _weight_only_check(got, x, w, scale, zp, bias, dtype):
    """|error| <= accumulation bound: products are exact in f32 (half activations; f32 ones
    enter as two halves, 2^-21 relative -- or 2^-25 absolute per activation where the low
    half is a subnormal half, i.e. for |x| < 1/8), the f32 accumulation of K terms adds
    K * 2^-24 of sum |x||w|, then one rounding to the output type."""
    want, bound = O.weight_only_qgemm(x, w, scale, zp, bias)
    k = x.shape[1]
    tol = bound * (k * 2.0 ** -24 + 2.0 ** -20) + 1e-30
    if dtype == torch.float32:
        _, wsum = O.weight_only_qgemm(np.ones((1, k), np.float32), w, scale, zp, None)
        tol = tol + wsum * 2.0 ** -25
    tol = tol + (np.abs(want) + bound * 2.0 ** -12) * (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -22)
    err = np.abs(host(got).astype(np.float64) - want)
    assert (err <= tol).all(), "max excess %.3g at %s" % (float((err - tol).max()),
                                                          np.unravel_index(np.argmax(err - tol), err.shape))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("k,n", [(768, 768), (768, 3072), (3072, 768)])
@pytest.mark.parametrize("m", [1, 16, 128, 1024])
def test_weight_only_qgemm_bert_linears(K, m, k, n, dtype):
    """Weight-only quantized linear on the BERT-base shapes: uint8 weights with per-channel
    scale and zero point near 128 (the reference pattern's quantization), bias, f16 and f32
    activations, every kernel form (small-M, both tile shapes)."""
    rng = np.random.default_rng(m * 7 + k + n)
    x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed=False)
    got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), dev(bias))
    assert got.dtype == dtype and tuple(got.shape) == (m, n)
    _weight_only_check(got, x, w, scale, zp, bias, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("signed", [False, True])
@pytest.mark.parametrize("m", [2, 24, 200])
def test_weight_only_qgemm_zero_points_at_the_documented_extremes(K, dtype, signed, m):
    """Zero points at both ends of the documented range (uint8 weights [-1024, 1024], int8
    weights [-1152, 896]), odd values next to the ends included: the kernels' half 1024 + zp
    (+ 128) is exact there, so the usual accumulation bound holds."""
    k, n = 256, 96
    rng = np.random.default_rng(m + int(signed))
    x, w, scale, _, bias = _weight_only_case(rng, m, k, n, dtype, signed)
    lo, hi = (-1152, 896) if signed else (-1024, 1024)
    ends = np.array([lo, lo + 1, lo + 3, hi - 3, hi - 1, hi], np.int32)
    zp = ends[rng.integers(0, len(ends), n)]
    zp[:len(ends)] = ends
    scale = (scale / 8).astype(scale.dtype)              # keeps f16 results finite
    got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), dev(bias))
    _weight_only_check(got, x, w, scale, zp, bias, dtype)


@pytest.mark.parametrize("k,n", [(64, 4), (128, 8), (192, 20), (1280, 200), (4096, 4096),
                                 (11008, 4096)])
def test_weight_only_undo_compiler_layout(K, k, n):
    """The inverse of the compiler's constant-weight permutation
    (R tao_compiler/mlir/disc/transforms/disc_transform_weight_data_layout_for_weight_only_gemm.cc
    :54-300, :362-370), bit for bit against the oracle's restatement of the four functions."""
    from oracle import weight_layout_oracle as WL
    w_kn = np.random.default_rng(k + n).integers(0, 256, (k, n), dtype=np.uint8)
    got = K.weight_only_undo_compiler_layout(dev(WL.forward(w_kn)))
    assert tuple(got.shape) == (n, k)
    np.testing.assert_array_equal(host(got), w_kn.T)


def test_weight_only_undo_compiler_layout_refuses_shapes_outside_the_pass_domain(K):
    for k, n in [(96, 8), (64, 6)]:
        with pytest.raises(RuntimeError, match="K % 64 == 0"):
            K.weight_only_undo_compiler_layout(torch.zeros((k, n), dtype=torch.uint8, device="cuda"))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_weight_only_qgemm_layouts_and_ragged_shapes(K, dtype):
    """[K,N] weights as the custom call passes them (with and without the scratch for the
    transpose), int8 weights, no bias / no zero points, shapes that leave partial tiles, a k
    depth that is not a multiple of 32, and the shapes the alignment rules send to the
    kernel without them (the reference's own test uses K = 3, N = 5)."""
    rng = np.random.default_rng(77)
    for (m, k, n) in [(2, 3, 5), (33, 48, 40), (200, 80, 136), (1, 16, 1), (70, 2064, 100),
                      (130, 40, 260), (5, 1000, 33),
                      # enough 128 x 128 tiles for the kernel that stages both operands in LDS:
                      # ragged last tiles in M and N, k depths off a multiple of 64
                      (1500, 80, 1100), (1290, 208, 1300), (9, 4112, 40),
                      # a full round of 256 x 256 tiles (ragged last row and column of tiles,
                      # XCD-ordered) and of 256 x 128 tiles
                      (4000, 144, 4090), (2000, 80, 4090)]:
        for signed in (False, True):
            x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed)
            got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), dev(bias))
            _weight_only_check(got, x, w, scale, zp, bias, dtype)
            w_kn = np.ascontiguousarray(w.T)
            for ws in (True, False):
                got = K.weight_only_qgemm(dev(x), dev(w_kn), dev(scale), dev(zp), None, tp_b=False,
                                          workspace=ws)
                _weight_only_check(got, x, w, scale, zp, None, dtype)
            got = K.weight_only_qgemm(dev(x), dev(w), dev(scale))
            _weight_only_check(got, x, w, scale, None, None, dtype)
    # small-magnitude f32 activations: the low halves are subnormal, the absolute term of the
    # bound takes over
    if dtype == torch.float32:
        x, w, scale, zp, bias = _weight_only_case(rng, 40, 256, 96, dtype, False)
        x = (x * 1e-4).astype(np.float32)
        got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), None)
        _weight_only_check(got, x, w, scale, zp, None, dtype)
    # strided activations (a column slice of a wider tensor)
    x, w, scale, zp, bias = _weight_only_case(rng, 64, 64, 96, dtype, False)
    wide = dev(np.concatenate([x, x], axis=1))
    got = K.weight_only_qgemm(wide[:, :64], dev(w), dev(scale), dev(zp), dev(bias))
    _weight_only_check(got, x, w, scale, zp, bias, dtype)
    empty = K.weight_only_qgemm(dev(x[:0]), dev(w), dev(scale), dev(zp), dev(bias))
    assert tuple(empty.shape) == (0, 96)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_weight_only_qgemm_one_or_two_rows(K, dtype):
    """One or two activation rows (three or four against narrow weights): the row-streaming
    kernel on the vector ALUs (k depths that end inside a wave's 1 KiB step and inside a group
    of steps, N that ends inside a workgroup's 8 channels, signed weights, strided activations,
    no bias / zero points), and a k depth whose rows do not fit the LDS, which the matrix-core
    kernels take."""
    rng = np.random.default_rng(1234)
    for (m, k, n, signed) in [(1, 16, 1, False), (1, 768, 3072, False), (1, 4096, 100, True),
                              (2, 2064, 77, False), (1, 8192 + 48, 19, False), (2, 8192, 64, True),
                              (1, 1024 * 5 + 16, 9, False), (1, 40000, 24, False), (2, 20000, 24, False),
                              (3, 3072, 768, False), (4, 2064, 77, True), (4, 8192 + 48, 1024, False),
                              (3, 16384, 20, False), (4, 2048, 1030, False)]:
        x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed)
        got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), dev(bias))
        _weight_only_check(got, x, w, scale, zp, bias, dtype)
        wide = dev(np.concatenate([x, x], axis=1))
        got = K.weight_only_qgemm(wide[:, :k], dev(w), dev(scale))
        _weight_only_check(got, x, w, scale, None, None, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_weight_only_qgemm_small_m_staged_through_lds(K, dtype):
    """5 .. 32 rows against deep weights: the kernel that stages both operands through
    wave-private LDS (16 and 32 staged rows; k depths that end inside a unit of 64 and inside
    a group of three units; N that ends inside a workgroup's 32 channels; signed weights; few
    rows against 8192 channels and more, where it starts at five rows whatever the depth).
    With f32 activations it ends at 16 rows and the tiled kernel takes the rest."""
    rng = np.random.default_rng(99)
    for (m, k, n, signed) in [(12, 2048, 96, False), (16, 3072, 768, False), (17, 2064, 100, True),
                              (32, 4096, 330, False), (5, 6160, 72, True), (9, 8192, 64, False),
                              (31, 2048 + 16 * 9, 40, False), (7, 2048, 8200, False)]:
        x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed)
        got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), dev(bias))
        _weight_only_check(got, x, w, scale, zp, bias, dtype)
        # strided activations and no bias / zero points
        wide = dev(np.concatenate([x, x], axis=1))
        got = K.weight_only_qgemm(wide[:, :k], dev(w), dev(scale))
        _weight_only_check(got, x, w, scale, None, None, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_weight_only_qgemm_split_over_k(K, dtype):
    """M between the skinny kernels' range and the sizes whose tiles fill the chip: the launch
    is split over k (f32 partial sums in the scratch, a reduction launch behind the GEMM).
    Ragged M, N and k ranges, N that is not a multiple of 4 (scalar reduction), with and
    without the scratch (without it the unsplit kernels run), the same bits on every call, and
    a caller-owned scratch that is reused."""
    import bladedisc_amd._lib as _lib
    L = _lib.lib()
    rng = np.random.default_rng(4242)
    code = 1 if dtype == torch.float16 else 0
    split_seen = 0
    for (m, k, n) in [(33, 1024, 256), (64, 3072, 768), (100, 2064, 130), (128, 4096, 1024),
                      (200, 1040, 333), (512, 2048, 640), (48, 1536, 4096), (70, 4112, 520),
                      (40, 3600, 203)]:
        x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed=False)
        plain = L.dq8_weight_only_qgemm_workspace_bytes(n, k, 1)
        need = L.dq8_weight_only_qgemm_workspace_bytes_ex(m, n, k, 1, code)
        splits = _weight_only_plan(m, n, k, dtype)[1]
        assert plain == 0 and need == (4 * m * n * splits if splits > 1 else 0)
        split_seen += splits > 1
        args = (dev(x), dev(w), dev(scale), dev(zp), dev(bias))
        got = K.weight_only_qgemm(*args)
        _weight_only_check(got, x, w, scale, zp, bias, dtype)
        again = K.weight_only_qgemm(*args)
        assert torch.equal(got, again)
        unsplit = K.weight_only_qgemm(*args, workspace=False)
        _weight_only_check(unsplit, x, w, scale, zp, bias, dtype)
        if need:
            ws = torch.empty(need + 4096, dtype=torch.uint8, device="cuda")
            ws.fill_(0xff)                                   # (NaN patterns: nothing may leak)
            assert torch.equal(K.weight_only_qgemm(*args, workspace=ws), got)
            assert bool((ws[:need].view(torch.int32) != -1).any()) and bool((ws[need:] == 0xff).all())
            assert torch.equal(K.weight_only_qgemm(*args, workspace=ws), got)
            # a scratch that is too small for the partial sums: the unsplit kernels
            assert torch.equal(K.weight_only_qgemm(*args, workspace=ws[:need - 16]), unsplit)
        # [K,N] weights: the transposed copy and the partial sums share the scratch
        got_kn = K.weight_only_qgemm(dev(x), dev(np.ascontiguousarray(w.T)), dev(scale), dev(zp),
                                     dev(bias), tp_b=False)
        assert torch.equal(got_kn, got)
    assert split_seen >= 5


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_weight_only_qgemm_few_rounds_of_small_tiles(K, dtype):
    """Above 32 rows while the tiles are a few rounds of the chip: 64 x 64 tiles on four waves
    (or 128 x 128), over the whole k range where a split is not estimated to pay -- shallow k,
    ragged M and N, a k range that is not a multiple of the 64-deep tile, M on both sides of
    the tile sizes."""
    import bladedisc_amd._lib as _lib
    L = _lib.lib()
    rng = np.random.default_rng(5151)
    code = 1 if dtype == torch.float16 else 0
    unsplit_seen = 0
    for (m, k, n) in [(33, 16, 64), (40, 256, 1024), (64, 272, 100), (65, 768, 3072),
                      (128, 768, 768), (129, 528, 200), (300, 1024, 4096), (700, 784, 1000),
                      (1000, 768, 3072)]:
        x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed=bool(m & 1))
        unsplit_seen += L.dq8_weight_only_qgemm_workspace_bytes_ex(m, n, k, 1, code) == 0
        args = (dev(x), dev(w), dev(scale), dev(zp), dev(bias))
        got = K.weight_only_qgemm(*args)
        _weight_only_check(got, x, w, scale, zp, bias, dtype)
        assert torch.equal(K.weight_only_qgemm(*args), got)
        _weight_only_check(K.weight_only_qgemm(*args, workspace=False), x, w, scale, zp, bias, dtype)
    assert unsplit_seen >= 5


@pytest.mark.parametrize("dtype,m,k,n,signed", [
    # 32 x 64 tiles: one k tile, shorter than 128; fewer k tiles than LDS stages; a split whose last
    # k range is a part of a tile
    (torch.float16, 33, 80, 17, False), (torch.float16, 102, 384, 65, True), (torch.float16, 85, 1888, 25, False),
    # 64 x 64, 64 x 128, 128 x 128 (four and eight waves), 128 x 256: a part of a row and of a channel
    # tile, k ending inside a k tile
    (torch.float16, 292, 656, 1771, False), (torch.float16, 265, 656, 3662, True),
    (torch.float16, 323, 672, 5777, False), (torch.float16, 274, 1936, 6689, True),
    (torch.float16, 978, 1072, 4133, False),
    (torch.float32, 45, 16, 27, True), (torch.float32, 58, 1312, 19, False), (torch.float32, 68, 144, 5877, False),
    (torch.float32, 1425, 48, 671, True), (torch.float32, 1375, 560, 651, False),
    (torch.float32, 356, 752, 5530, True)])
def test_weight_only_qgemm_tiles_loaded_into_lds(K, dtype, m, k, n, signed):
    """Every tile form of the kernel that loads both operands straight into LDS, at sizes its tiles do
    not divide, with results whose rows start off 16 bytes and nothing written beside them; activations
    and weights past the rows and the k range are NaN / 255, so that nothing outside may be used."""
    rng = np.random.default_rng(m + k + n)
    x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed)
    wide_x, wide_w = _weight_only_framed(x, w, dtype, signed)
    splits = _weight_only_plan(m, n, k, dtype)[1]
    ws = torch.empty(max(4 * m * n * splits, 16), dtype=torch.uint8, device="cuda")
    frame = torch.full((m + 1, n + 5), 7.0, dtype=dtype, device="cuda")
    out = frame[:m, 1:n + 1]
    _weight_only_raw(wide_x, wide_w, dev(scale), dev(zp), dev(bias), out, ws, ws.nbytes)
    _weight_only_check(out, x, w, scale, zp, bias, dtype)
    assert bool((frame[:, 0] == 7).all()) and bool((frame[:, n + 1:] == 7).all()) and bool((frame[m] == 7).all())
    got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), workspace=False)
    _weight_only_check(got, x, w, scale, None, None, dtype)


@pytest.mark.parametrize("dtype,m,k,n,form,splits", [
    (torch.float16, 33, 2064, 34, 0, 7), (torch.float16, 34, 7568, 1377, 1, 8), (torch.float16, 36, 7968, 4134, 2, 6),
    (torch.float16, 66, 6240, 5481, 3, 4), (torch.float16, 129, 5456, 6579, 4, 2),
    (torch.float16, 259, 7856, 6602, 5, 3),
    (torch.float32, 33, 2096, 33, 6, 7), (torch.float32, 33, 2192, 2727, 7, 4), (torch.float32, 67, 6640, 5523, 8, 8),
    (torch.float32, 33, 4752, 5469, 9, 4), (torch.float32, 66, 7344, 5614, 10, 4),
    # rows off 16 bytes
    (torch.float16, 33, 1131, 33, 11, 4), (torch.float16, 67, 4763, 4230, 12, 6)])
def test_weight_only_qgemm_every_tile_form_split_over_k(K, dtype, m, k, n, form, splits):
    """Every tile form with the k range split (the form and the ranges are asserted): M and N off the
    tile, ranges that begin at odd multiples of 64, a last range that ends inside a k tile, operands in
    frames of NaN / 255, a scratch of exactly the partial sums, filled with NaN patterns, and nothing
    written behind it or beside the results."""
    ragged = k % 16 != 0
    assert _weight_only_plan(m, n, k, dtype, ragged) == (form, splits)
    rng = np.random.default_rng(m + k + n)
    x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed=bool(form & 1))
    wide_x, wide_w = _weight_only_framed(x, w, dtype, bool(form & 1))
    need = 4 * m * n * splits
    ws = torch.full((need + 4096,), 0xff, dtype=torch.uint8, device="cuda")
    frame = torch.full((m + 1, n + 5), 7.0, dtype=dtype, device="cuda")
    out = frame[:m, 1:n + 1]
    _weight_only_raw(wide_x, wide_w, dev(scale), dev(zp), dev(bias), out, ws, need)
    _weight_only_check(out, x, w, scale, zp, bias, dtype)
    assert bool((frame[:, 0] == 7).all()) and bool((frame[:, n + 1:] == 7).all()) and bool((frame[m] == 7).all())
    assert bool((ws[need:] == 0xff).all())
    planes = ws[:need].view(torch.float32).reshape(splits, m, n)
    assert bool(torch.isfinite(planes).all())
    first = out.clone()
    _weight_only_raw(wide_x, wide_w, dev(scale), dev(zp), dev(bias), out, ws, need)
    assert torch.equal(out, first)


@pytest.mark.parametrize("m,k,n,form,splits", [
    (35, 72, 140, 0, 1), (42, 1868, 32, 0, 8), (92, 2700, 105, 0, 8), (227, 412, 2227, 1, 1), (1018, 68, 1282, 2, 1),
    (286, 216, 4074, 2, 1), (1727, 280, 3699, 3, 1), (1030, 4100, 4090, 5, 1), (1021, 4100, 4090, 4, 1),
    (66, 6236, 2481, 0, 2)])
@pytest.mark.parametrize("signed", [False, True])
def test_weight_only_qgemm_rows_that_begin_on_four_bytes(K, m, k, n, form, splits, signed):
    """Rows of whole words on the tiles of aligned rows: 4, 8 and 12 k in the last group of 16, in each half of a
    unit, a last range of 4 to 12 k (92 x 2700), in frames of NaN / 255, with the scratch that is asked for."""
    assert _weight_only_plan(m, n, k, torch.float16) == (form, splits)
    rng = np.random.default_rng(m + k + n)
    x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, torch.float16, signed)
    wide_x, wide_w = _weight_only_framed(x, w, torch.float16, signed)
    ws = torch.full((4 * m * n * 8,), 0xff, dtype=torch.uint8, device="cuda")
    frame = torch.full((m + 1, n + 5), 7.0, dtype=torch.float16, device="cuda")
    out = frame[:m, 1:n + 1]
    _weight_only_raw(wide_x, wide_w, dev(scale), dev(zp), dev(bias), out, ws, ws.nbytes)
    _weight_only_check(out, x, w, scale, zp, bias, torch.float16)
    assert bool((frame[:, 0] == 7).all()) and bool((frame[:, n + 1:] == 7).all()) and bool((frame[m] == 7).all())
    for workspace in (True, False):
        got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), zero_points=dev(zp), workspace=workspace)
        _weight_only_check(got, x, w, scale, zp, None, torch.float16)


@pytest.mark.parametrize("m,k,n,signed", [
    (17, 400, 4097, False), (24, 1040, 4111, True), (32, 2048, 5000, False), (31, 784, 6161, True),
    (17, 2816, 6144, False), (25, 1024, 8177, True), (32, 2064, 8192, False), (20, 384, 4097, True),
    (32, 2832, 8192, False), (29, 512, 8193, True), (18, 2064, 4096, False)])
def test_weight_only_qgemm_f32_rows_on_either_side_of_the_tiles_line(K, m, k, n, signed):
    """17 to 32 rows of f32 on 32-channel workgroups of the staged kernel (low halves on sums of their own,
    the waves' sums in pairs) and on tiles, at the edges of the rule between them, in frames of NaN / 255."""
    rng = np.random.default_rng(m + k + n)
    x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, torch.float32, signed)
    wide_x, wide_w = _weight_only_framed(x, w, torch.float32, signed)
    splits = _weight_only_plan(m, n, k, torch.float32)[1]
    ws = torch.empty(max(4 * m * n * splits, 16), dtype=torch.uint8, device="cuda")
    frame = torch.full((m + 1, n + 5), 7.0, device="cuda")
    out = frame[:m, 1:n + 1]
    _weight_only_raw(wide_x, wide_w, dev(scale), dev(zp), dev(bias), out, ws, ws.nbytes)
    _weight_only_check(out, x, w, scale, zp, bias, torch.float32)
    assert bool((frame[:, 0] == 7).all()) and bool((frame[:, n + 1:] == 7).all()) and bool((frame[m] == 7).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_weight_only_qgemm_strided_rows_in_and_out(K, dtype):
    """Activation and result rows that are slices of wider buffers (ldx > K, ldo > N), one shape
    per kernel family (row-streaming, 16-channel, staged, 64 x 64 tiles unsplit and split over
    k, 128-row and 256-row tiles): right results, and nothing written outside the slice."""
    rng = np.random.default_rng(5)
    for (m, k, n) in [(1, 4096, 100), (4, 3072, 768), (8, 768, 200), (8, 2048, 8200),
                      (24, 2064, 300), (40, 4096, 520), (100, 784, 200), (300, 1024, 1000),
                      (64, 8192, 264), (1000, 768, 3072), (2100, 256, 520)]:
        x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, False)
        wide = dev(np.concatenate([x, x], axis=1))
        frame = torch.full((m, n + 24), 7.0, dtype=dtype, device="cuda")
        out = frame[:, 8:8 + n]
        K.weight_only_qgemm(wide[:, :k], dev(w), dev(scale), dev(zp), dev(bias), out=out)
        _weight_only_check(out, x, w, scale, zp, bias, dtype)
        assert bool((frame[:, :8] == 7).all()) and bool((frame[:, 8 + n:] == 7).all())


def test_weight_only_dispatch_sweep_stays_within_the_accumulation_bound(K):
    """Seeded sweep over what the launcher's choice depends on -- rows from 1 to several rounds
    of tiles, k from one 16-chunk to 9000, narrow to wide weights, both activation types,
    signed and unsigned weights: whichever kernel the rules and the cost estimate land on,
    the result stays within the accumulation bound of the oracle."""
    rng = np.random.default_rng(20260202)
    ms = [1, 2, 3, 4, 5, 8, 9, 12, 16, 17, 24, 31, 32, 33, 48, 64, 65, 100, 128, 129, 200, 256,
          300, 512, 700, 1100]
    cases = []
    for m in ms:
        for _ in range(2):
            k = 16 * int(rng.integers(1, 560))
            n = int(rng.integers(1, 3000))
            while m * k * n > 1.2e9:
                n = max(1, n // 2)
            cases.append((m, k, n))
    # few rows against wide weights, deep k against narrow ones
    cases += [(5, 2048, 8200), (11, 2064, 9000), (24, 2048, 8192), (4, 8192, 1000),
              (3, 2048, 1024), (24, 1536, 1536), (40, 8192, 520), (2100, 256, 4100)]
    for i, (m, k, n) in enumerate(cases):
        dtype = torch.float16 if i % 2 == 0 else torch.float32
        x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed=bool(i % 3 == 0))
        got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), dev(bias))
        _weight_only_check(got, x, w, scale, zp, bias, dtype)


def test_multi_kernel_paths_replay_from_a_captured_graph(K):
    """The paths that are several launches -- a weight-only GEMM split over k (GEMM, then the
    reduction), a stem convolution through space to depth (two re-layouts, then the
    convolution) -- captured into one HIP graph with caller-owned scratch and replayed with
    other work in between: every replay gives the eager result, also after the inputs change."""
    import bladedisc_amd._lib as _lib
    L = _lib.lib()
    rng = np.random.default_rng(808)
    m, k, n = 64, 3072, 768
    assert _weight_only_plan(m, n, k, torch.float16)[1] > 1
    x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, torch.float16, False)
    xd, wd, sd, zd, bd = dev(x), dev(w), dev(scale), dev(zp), dev(bias)
    need = L.dq8_weight_only_qgemm_workspace_bytes_ex(m, n, k, 1, 1)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    out = torch.empty((m, n), dtype=torch.float16, device="cuda")
    ci, co, h = 3, 32, 40
    cx = dev(rng.integers(-128, 128, (2, h, h, ci), dtype=np.int8))
    cw = dev(rng.integers(-128, 128, (co, 7, 7, ci), dtype=np.int8))
    md = list(O.NHWC_OHWI_METADATA) + [2, 2, 1, 1, 1]
    osh = [2, h // 2, h // 2, co]
    cout = torch.empty(tuple(osh), dtype=torch.int32, device="cuda")

    def run():
        K.weight_only_qgemm(xd, wd, sd, zd, bd, out=out, workspace=ws)
        K.qconv2d(cx, cw, [3, 3, 3, 3], md, osh, K.EPI_ACC_S32, out=cout)

    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        run()
    for rep in range(4):
        if rep == 2:                                       # new inputs in the captured buffers
            xd.copy_(dev(rng.standard_normal((m, k)).astype(np.float16)))
            cx.copy_(dev(rng.integers(-128, 128, (2, h, h, ci), dtype=np.int8)))
        out.zero_()
        cout.zero_()
        ws.fill_(0xff)
        graph.replay()
        torch.cuda.synchronize()
        got, cgot = out.clone(), cout.clone()
        want = K.weight_only_qgemm(xd, wd, sd, zd, bd)
        cwant = K.qconv2d(cx, cw, [3, 3, 3, 3], md, osh, K.EPI_ACC_S32)
        assert torch.equal(got, want), rep
        assert torch.equal(cgot, cwant), rep


def test_dispatch_sweep_agrees_with_the_generic_kernel(K):
    """Seeded sweep over what the library's own choice of kernel depends on -- M from one row
    to several rounds of the largest tiles, N, K, the epilogue family, fused operators -- with
    the scalar generic kernel (variant 0, itself pinned against the oracle above) as the
    yardstick on the same device buffers: every combination must give the same bits, whichever
    kernel the heuristic lands on (row-streaming for one or two rows against deep weights,
    small-M, 64 / 128 / 256-wide tiles, persistent forms)."""
    rng = np.random.default_rng(20260101)
    ms = [1, 7, 16, 31, 33, 100, 500, 1000, 2100, 4096, 9000, 20000]
    cases = 0
    # (m, n, k): three random (n, k) per m, then one and two rows against rows of 2048 of k and
    # more, with k ending inside a wave's step and N inside a workgroup's channels, then few
    # rows against weights wide enough for the tiled kernel to take them, then k deep enough
    # for the split over four wave groups
    shapes = [(m, None, None) for m in ms for _ in range(3)] + \
             [(1, 100, 3072), (2, 9, 2048), (1, 40, 8208), (2, 130, 4112),
              (3, 14400, 2048), (9, 9250, 2064), (16, 9216, 2048), (8, 9216, 2048),
              (40, 1000, 8192), (100, 520, 8208),
              # the small-M kernel's range above 32 rows: one, two and four row tiles per
              # workgroup, ragged N and k, partial last row tile
              (64, 776, 784), (130, 40, 3088), (256, 768, 768), (200, 24, 2064),
              (64, 4096, 4096), (33, 4104, 4096), (250, 72, 1040)]
    for m, n_fixed, k_fixed in shapes:
        if True:
            n = n_fixed or int(rng.choice([16, 48, 64, 136, 768, 1024, 2304, 3072]))
            k = k_fixed or int(rng.choice([16, 64, 144, 768, 1040, 3072]))
            if m * n * k > 2.2e10:
                k = 64
            a = dev(rng.integers(-128, 128, (m, k), dtype=np.int8))
            w = dev(rng.integers(-128, 128, (n, k), dtype=np.int8))
            sx = dev(np.array([rng.uniform(0.01, 0.03)], np.float32))
            sw = dev(rng.uniform(0.001, 0.05, n).astype(np.float32))
            so = dev(np.array([float(np.sqrt(k)) * 0.02 * 0.025 * 5400 / 40.0], np.float32))
            bf = dev((rng.standard_normal(n) * 3).astype(np.float32))
            b32 = dev(rng.integers(-20000, 20000, n).astype(np.int32))
            table = dev(rng.integers(-128, 128, 256, dtype=np.int8))
            resid = dev(rng.integers(-128, 128, (m, n), dtype=np.int8))
            rs = dev(np.array([0.05], np.float32))
            s2 = dev(np.array([0.07], np.float32))
            sc = dict(sx=sx, sw=sw, so=so)
            plans = [
                (K.EPI_ACC_S32, {}, None),
                (K.EPI_REQUANT_CPU, dict(bias=bf, zo=2, **sc), None),
                (K.EPI_REQUANT_GPU, dict(bias=bf, **sc), None),
                (K.EPI_DEQUANT_F32, dict(sx=sx, sw=sw, bias=bf), None),
                (K.EPI_REQUANT_CPU_DEQUANT_F32, dict(bias=bf, zo=2, **sc), None),
                (K.EPI_REQUANT_FIXEDPOINT, dict(bias=b32, zo=-1, **sc), None),
                (K.EPI_REQUANT_CPU, dict(bias=bf, **sc), dict(table=table)),
                (K.EPI_REQUANT_GPU, dict(bias=bf, **sc),
                 dict(residual=resid, residual_scale=rs, residual_zp=3, relu=True, out_scale=s2, out_zp=-4)),
            ]
            for epi, kw, post in plans:
                if post is None:
                    want = K.qgemm(a, w, epi, variant=0, **kw)
                    got = K.qgemm(a, w, epi, **kw)
                else:
                    # (fused operators go with the library's own choice: the yardstick is the chain
                    # of separate calls on the generic kernel's result)
                    q = K.qgemm(a, w, epi, variant=0, **kw)
                    if "table" in post:
                        want = K.lut8(q, table)
                    else:
                        zero = torch.zeros(1, dtype=torch.int32, device="cuda")
                        t = K.dequantize(q, so, zero) + K.dequantize(
                            resid, rs, torch.full((1,), 3, dtype=torch.int32, device="cuda"))
                        t = torch.where(t < 0, torch.zeros_like(t), t)
                        want = K.quantize(t, s2, torch.full((1,), -4, dtype=torch.int32, device="cuda"))
                    got = K.qgemm(a, w, epi, post=K.make_postops(**post), **kw)
                assert got.dtype == want.dtype
                same = torch.equal(got.view(torch.int32) if got.dtype == torch.float32 else got,
                                   want.view(torch.int32) if want.dtype == torch.float32 else want)
                assert same, (m, n, k, epi, post)
                cases += 1
    assert cases == len(shapes) * 8


def test_conv_dispatch_sweep_agrees_with_the_generic_kernel(K):
    """The same for convolutions: batch, image size, channel counts (multiples of 16 and not),
    filter, stride, padding and dilation drawn from a seeded generator; the library's choice
    (direct 3x3 kernels, implicit GEMM tiles, 1x1 as a plain GEMM, channel padding through the
    scratch) against the generic kernel, for the int8, int32, f32 and fixed-point results and a
    fused table."""
    rng = np.random.default_rng(20260102)
    cases = 0
    shapes = []
    for _ in range(30):
        nb = int(rng.choice([1, 2, 8, 32, 70]))
        h = int(rng.choice([7, 14, 28, 33, 56]))
        w_ = int(rng.choice([7, 14, 28, 30, 56]))
        ci = int(rng.choice([3, 16, 24, 32, 64, 128, 256]))
        co = int(rng.choice([16, 40, 64, 128, 256]))
        k = int(rng.choice([1, 3, 3, 5]))
        stride = int(rng.choice([1, 1, 2]))
        dil = int(rng.choice([1, 1, 2]))
        pad = int(rng.integers(0, 3))
        shapes.append((nb, h, w_, ci, co, k, stride, dil, pad))
    # k deep enough for the 64 x 64 tiles to split it over four wave groups
    shapes += [(8, 7, 7, 1024, 256, 3, 1, 1, 1), (1, 10, 10, 1040, 70, 3, 1, 1, 0)]
    for (nb, h, w_, ci, co, k, stride, dil, pad) in shapes:
        ho = (h + 2 * pad - dil * (k - 1) - 1) // stride + 1
        wo = (w_ + 2 * pad - dil * (k - 1) - 1) // stride + 1
        if ho <= 0 or wo <= 0 or nb * ho * wo * co * k * k * ci > 6e10:
            continue
        x = dev(rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8))
        wt = dev(rng.integers(-128, 128, (co, k, k, ci), dtype=np.int8))
        md = list(O.NHWC_OHWI_METADATA) + [stride, stride, dil, dil, 1]
        padding, osh = [pad] * 4, [nb, ho, wo, co]
        sc = dict(sx=dev(np.array([0.02], np.float32)), sw=dev(rng.uniform(0.001, 0.05, co).astype(np.float32)),
                  so=dev(np.array([float(np.sqrt(k * k * ci)) * 0.02 * 0.025 * 5400 / 40.0], np.float32)))
        b32 = dev(rng.integers(-20000, 20000, co).astype(np.int32))
        table = dev(rng.integers(-128, 128, 256, dtype=np.int8))
        for epi, kw in ((K.EPI_ACC_S32, {}), (K.EPI_REQUANT_CPU, dict(zo=1, **sc)),
                        (K.EPI_REQUANT_CPU_DEQUANT_F32, sc), (K.EPI_REQUANT_FIXEDPOINT, dict(bias=b32, **sc))):
            want = K.qconv2d(x, wt, padding, md, osh, epi, variant=0, **kw)
            got = K.qconv2d(x, wt, padding, md, osh, epi, **kw)
            v = (lambda t: t.view(torch.int32) if t.dtype == torch.float32 else t)
            assert torch.equal(v(got), v(want)), (nb, h, w_, ci, co, k, stride, pad, dil, epi)
            cases += 1
        q = K.qconv2d(x, wt, padding, md, osh, K.EPI_REQUANT_CPU, variant=0, **sc)
        got = K.qconv2d(x, wt, padding, md, osh, K.EPI_REQUANT_CPU, **sc, post=K.make_postops(table=table))
        assert torch.equal(got, K.lut8(q, table)), (nb, h, w_, ci, co, k, stride, pad, dil)
    assert cases >= 80


@pytest.mark.parametrize("nb,h,ci,co,k", [(1, 9, 64, 64, 3), (5, 31, 64, 64, 3), (3, 17, 128, 48, 3),
                                          (2, 56, 64, 256, 1), (40, 33, 64, 48, 1), (8, 33, 128, 512, 1),
                                          (9, 28, 256, 64, 1), (9, 28, 256, 128, 1), (2, 14, 512, 2048, 1),
                                          (3, 28, 16, 64, 4), (1, 7, 512, 192, 3)])
def test_clamping_tables_and_int8_residuals_equal_the_separate_operators(K, nb, h, ci, co, k):
    """A fused table that clamps (ReLU, ReLU6) is taken as bounds, an int8 residual runs on the
    accumulators where the scales allow it: the bits of the separate calls, with and without
    zero points, with scales and tables on either side of those conditions."""
    rng = np.random.default_rng(h * ci + co)
    pad = [k // 2, (k - 1) // 2] * 2
    x = dev(rng.integers(-128, 128, (nb, h, h, ci), dtype=np.int8))
    wt = dev(rng.integers(-128, 128, (co, k, k, ci), dtype=np.int8))
    md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
    osh = [nb, h, h, co]
    s_acc = float(np.sqrt(k * k * ci) * 74 * 74)
    so = np.float32(0.043)
    sc = dict(sx=dev(np.array([0.02], np.float32)), so=dev(np.array([so])),
              sw=dev((rng.uniform(0.7, 1.3, co) * (50 * 0.043 / 0.02 / s_acc)).astype(np.float32)))
    bias = dev((rng.standard_normal(co) * 20 * so).astype(np.float32))
    zi = lambda v: torch.full((1,), v, dtype=torch.int32, device="cuda")  # noqa: E731
    rq = dev(rng.integers(-128, 128, osh, dtype=np.int8))
    entries = np.arange(256).astype(np.uint8).view(np.int8)
    almost = np.clip(entries, 0, 127)
    almost[200] += 1
    for epi, zo in ((K.EPI_REQUANT_CPU, 0), (K.EPI_REQUANT_CPU, 3), (K.EPI_REQUANT_GPU, 0)):
        kw = dict(bias=bias if epi == K.EPI_REQUANT_CPU else dev(rng.standard_normal(co).astype(np.float32) * 20),
                  zo=zo, **sc)
        q = K.qconv2d(x, wt, pad, md, osh, epi, **kw)
        for table in (np.clip(entries, 0, 127), np.clip(entries, -7, 90), entries, almost,
                      np.full(256, 5, np.int8), np.clip(entries, -128, -1)):
            t = dev(np.ascontiguousarray(table.astype(np.int8)))
            got = K.qconv2d(x, wt, pad, md, osh, epi, post=K.make_postops(table=t), **kw)
            assert torch.equal(got, K.lut8(q, t))
        y = K.dequantize(q, sc["so"], zi(zo))
        for rz, z2, s2, relu in ((0, 0, 0.05, True), (0, 0, 0.05, False), (-5, -128, 0.037, True),
                                 (4, 130, 0.05, True), (0, -140, 0.05, True), (0, 0, -0.05, True),
                                 (0, 7, 2e12, False)):
            rs, ds2 = dev(np.array([0.031], np.float32)), dev(np.array([s2], np.float32))
            t = y + K.dequantize(rq, rs, zi(rz))
            t = torch.where(t < 0, torch.zeros_like(t), t) if relu else t
            want = K.quantize(t, ds2, zi(z2))
            got = K.qconv2d(x, wt, pad, md, osh, epi, post=K.make_postops(
                residual=rq, residual_scale=rs, residual_zp=rz, relu=relu, out_scale=ds2, out_zp=z2), **kw)
            assert torch.equal(got, want), (epi, zo, rz, z2, s2, relu)


@pytest.mark.parametrize("nb,h,w,co", [(1, 1, 2, 16), (1, 5, 7, 80), (2, 33, 31, 272), (3, 97, 64, 256), (9, 61, 59, 144)])
def test_conv_1x1_64_behind_a_residual_in_paired_slices(K, nb, h, w, co):
    """1 x 1 filters on 64 channels with an int8 residual: 64-channel slices, two workgroups to a compute
    unit; slices and pixel tiles that end anywhere, one workgroup to several rounds of pairs, the f32
    residual and the general tail (a scale outside the fast range) in the same slices."""
    rng = np.random.default_rng(nb * h + co)
    md = list(O.NHWC_OHWI_METADATA) + [1, 1, 1, 1, 1]
    osh = [nb, h, w, co]
    x = dev(rng.integers(-128, 128, (nb, h, w, 64), dtype=np.int8))
    wt = dev(rng.integers(-128, 128, (co, 1, 1, 64), dtype=np.int8))
    one = lambda v: dev(np.array([v], np.float32))  # noqa: E731
    z = torch.zeros(1, dtype=torch.int32, device="cuda")
    kw = dict(sx=one(0.02), so=one(0.043), bias=dev((rng.standard_normal(co) * 0.9).astype(np.float32)),
              sw=dev((rng.uniform(0.7, 1.3, co) * (50 * 0.043 / 0.02 / (8 * 74 * 74))).astype(np.float32)))
    y = K.dequantize(K.qconv2d(x, wt, [0] * 4, md, osh, K.EPI_REQUANT_CPU, **kw), kw["so"], z)
    rq = dev(rng.integers(-128, 128, osh, dtype=np.int8))
    rf = dev((rng.standard_normal(osh) * 2).astype(np.float32))
    for res, rs, s2 in ((rq, 0.031, 0.05), (rq, 0.031, 2e12), (rf, None, 0.05)):
        post = K.make_postops(residual=res, residual_scale=None if rs is None else one(rs), relu=True, out_scale=one(s2))
        got = K.qconv2d(x, wt, [0] * 4, md, osh, K.EPI_REQUANT_CPU, post=post, **kw)
        t = y + (res if rs is None else K.dequantize(res, one(rs), z))
        assert torch.equal(got, K.quantize(torch.where(t < 0, torch.zeros_like(t), t), one(s2), z)), (rs, s2)


@pytest.mark.parametrize("m,k,n", [(1, 64, 17), (3, 65, 1), (16, 79, 33), (17, 1000, 130), (32, 2049, 515), (200, 127, 70),
                                   (256, 260, 129), (65, 1001, 1501), (300, 100, 257), (513, 333, 64), (777, 1000, 1501),
                                   (1030, 4097, 260), (2100, 200, 3001), (4200, 72, 2100)])
def test_qgemm_ragged_rows_and_results(K, m, k, n):
    """k, n, alignments and row strides that are multiples of nothing, with and without zero points
    and fused operators: small-M kernel on the rows as they are, tiled kernels on copied rows,
    results stored from rows that begin at any byte -- bit-exact against the scalar kernel."""
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    gen = 0
    wide_a = dev(rng.integers(-128, 128, (m, k + 5), dtype=np.int8))
    wide_w = dev(rng.integers(-128, 128, (n, k + 3), dtype=np.int8))
    out8 = torch.empty((m, n + 3), dtype=torch.int8, device="cuda")
    out32 = torch.empty((m, n + 1), dtype=torch.int32, device="cuda")
    so = np.float32(0.02 * 0.025 * 74.0 * 74.0 * np.sqrt(k) / 40.0)
    sc = dict(sx=dev(np.array([0.02], np.float32)), so=dev(np.array([so])),
              sw=dev(rng.uniform(0.001, 0.05, n).astype(np.float32)))
    bias = dev((rng.standard_normal(n) * 20 * so).astype(np.float32))
    for a, w in ((wide_a[:, :k].contiguous(), wide_w[:, :k].contiguous()), (wide_a[:, 3:3 + k], wide_w[:, 1:1 + k])):
        for zx, zw in ((0, 0), (-11, 0), (5, -3)):
            kw = dict(zx=zx, zw=zw)
            acc = K.qgemm(a, w, K.EPI_ACC_S32, variant=gen, **kw)
            assert torch.equal(K.qgemm(a, w, K.EPI_ACC_S32, **kw), acc)
            got = K.qgemm(a, w, K.EPI_ACC_S32, out=out32[:, 1:], **kw)
            assert torch.equal(got, acc)
            q = K.qgemm(a, w, K.EPI_REQUANT_CPU, bias=bias, zo=2, variant=gen, **sc, **kw)
            assert torch.equal(K.qgemm(a, w, K.EPI_REQUANT_CPU, bias=bias, zo=2, **sc, **kw), q)
            assert torch.equal(K.qgemm(a, w, K.EPI_REQUANT_CPU, bias=bias, zo=2, out=out8[:, 1:n + 1], **sc, **kw), q)
            y = K.qgemm(a, w, K.EPI_REQUANT_CPU_DEQUANT_F32, bias=bias, **sc, **kw)
            want = K.qgemm(a, w, K.EPI_REQUANT_CPU_DEQUANT_F32, bias=bias, variant=gen, **sc, **kw)
            assert torch.equal(y.view(torch.int32), want.view(torch.int32))
    table = dev(rng.integers(-128, 128, 256, dtype=np.int8))
    got = K.qgemm(a, w, K.EPI_REQUANT_CPU, bias=bias, zo=2, post=K.make_postops(table=table), **sc, **kw)
    assert torch.equal(got, K.lut8(q, table))
    res = dev((rng.standard_normal((m, n)) * 40 * so).astype(np.float32))
    got = K.qgemm(a, w, K.EPI_REQUANT_CPU_DEQUANT_F32, bias=bias, post=K.make_postops(residual=res), **sc, **kw)
    assert torch.equal(got.view(torch.int32), (y + res).view(torch.int32))


@pytest.mark.parametrize("shape,axis", [((1,), None), ((7,), None), ((1027,), None), ((3, 5), 1), ((4, 1), 1), ((9, 3), 1),
                                        ((1000, 3073), 1), ((5, 259), 1), ((6, 258), 1), ((7, 1025), 0), ((33, 5), 0),
                                        ((3, 6, 7), 1), ((2, 5, 1, 3), 2), ((1001, 33), 0)])
def test_quantize_any_size_type_and_alignment(K, shape, axis):
    """Sizes that are multiples of nothing, every quantized type, f16 input, bases at any element:
    the oracle's bits, both ways and fake-quantized."""
    rng = np.random.default_rng(sum(shape))
    n = 1 if axis is None else shape[axis]
    x = (rng.standard_normal(shape) * 50).astype(np.float32)
    for name, lo, hi in (("int8", -128, 127), ("uint8", 0, 255), ("int16", -32768, 32767), ("int32", -2**31, 2**31 - 1)):
        scale = rng.uniform(0.5, 1.5, n).astype(np.float32) * np.float32(2e-3 if name == "int16" else 1.0)
        zp = rng.integers(-5, 6, n).astype(np.int32) + (128 if name == "uint8" else 0)
        for xin in (x, x.astype(np.float16)):
            want = O.quantize(xin.astype(np.float32), scale, zp, axis=axis, qmin=lo, qmax=hi, dtype=np.dtype(name).type)
            base = torch.empty(x.size + 1, dtype=dev(xin).dtype, device="cuda")
            for dx in (dev(xin), base[1:].view(shape)):
                dx.copy_(dev(xin))
                got = K.quantize(dx, dev(scale), dev(zp), axis=axis, qmin=lo, qmax=hi, dtype=getattr(torch, name))
                np.testing.assert_array_equal(host(got), want)
        want_f = O.dequantize(want, scale, zp, axis=axis)
        np.testing.assert_array_equal(host(K.dequantize(got, dev(scale), dev(zp), axis=axis)), want_f)
        if name in ("int8", "uint8"):
            xf = dev(xin.astype(np.float32))
            np.testing.assert_array_equal(host(K.fake_quant(xf, dev(scale), dev(zp), axis=axis, qmin=lo, qmax=hi)), want_f)


@pytest.mark.parametrize("b,s,heads", [(1, 1, 1), (2, 8, 12), (3, 17, 2), (1, 49, 3), (2, 64, 1), (1, 65, 12), (2, 333, 5)])
def test_attention_equals_softmax_of_the_scores(K, b, s, heads):
    """Edges of the 16-query and 64-key tiles, against the same in f64; the fused quantize is the
    quantize of the f32 result."""
    qkv = torch.randn(b, s, 3 * heads * 64, generator=torch.Generator().manual_seed(s)) * 1.5
    q, k, v = (t.double().reshape(b, s, heads, 64).transpose(1, 2) for t in qkv.chunk(3, dim=-1))
    want = (torch.softmax(q @ k.transpose(2, 3) / 8.0, -1) @ v).transpose(1, 2).reshape(b, s, heads * 64)
    got = K.attention(qkv.cuda(), heads)
    torch.testing.assert_close(got.cpu().double(), want, rtol=1e-5, atol=1e-5)
    scale = torch.full((1,), 0.02, device="cuda")
    assert torch.equal(K.attention(qkv.cuda(), heads, scale), K.quantize(got, scale, torch.zeros(1, dtype=torch.int32, device="cuda")))


@pytest.mark.parametrize("b,s,heads", [(1, 1, 1), (2, 8, 12), (3, 17, 2), (1, 33, 3), (2, 64, 1), (1, 65, 12), (2, 97, 3), (2, 333, 5)])
@pytest.mark.parametrize("step", [0.02, 0.1, 20.0, 50.0, 1000.0])
def test_attention_of_an_int8_projection(K, b, s, heads, step):
    """Edges of the 16-query, 32- and 64-key tiles with codes of the whole range, a wide and a narrow
    softmax (scores up to 10 / up to 230) and the best key alone (up to 2e10), against the same in f64.  Bound:
    the scale's f32 square and product move a difference of scores d by 3 ulp, its rounding and the exponential's ulp come on top, and d above 25
    contributes nothing: 25 * 3 * 2^-24 + 2 * 2^-24 of each probability, twice (also in their sum), and
    s / 8 roundings of sums of values up to 128 * step: below 1e-5 of that."""
    g = torch.Generator().manual_seed(s)
    codes = torch.randint(-128, 128, (b, s, 3 * heads * 64), generator=g, dtype=torch.int8)
    codes[:, -1, -64:] = -128
    scale = torch.full((1,), step)
    q, k, v = (t.double().reshape(b, s, heads, 64).transpose(1, 2) for t in (codes.double() * scale.double()).chunk(3, dim=-1))
    want = (torch.softmax(q @ k.transpose(2, 3) / 8.0, -1) @ v).transpose(1, 2).reshape(b, s, heads * 64)
    got = K.attention(codes.cuda(), heads, qkv_scale=scale.cuda())
    assert got.isfinite().all()
    assert (got.cpu().double() - want).abs().max().item() <= 1e-5 * 128 * step
    out_scale = torch.full((1,), 0.02, device="cuda")
    zero = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert torch.equal(K.attention(codes.cuda(), heads, out_scale, float(scale)), K.quantize(got, out_scale, zero))
    # a scale that is not a number, or infinite: of 0 * inf and inf - inf; zero: all keys alike
    for bad in (float("nan"), float("inf")):
        assert K.attention(codes.cuda(), heads, None, bad).isnan().all()
    assert (K.attention(codes.cuda(), heads, None, 0.0) == 0).all()


@pytest.mark.parametrize("gap", [5, 17, 31, 60, 100, 120])
def test_attention_keeps_small_probabilities_of_an_int8_projection(K, gap):
    """One key takes all the weight and has values of zero; what the others, 2^-gap of it each, add up to, against
    f64.  Bound, relative: the scale's square, its factor and their product with the difference of scores are 3.5
    roundings of an exponent of -gap, 3.5 * ln 2 * gap; the exponential, the sums of 80 positive products and of
    80 probabilities, the division and the last product on top."""
    keys = 80
    g = torch.Generator().manual_seed(gap)
    q = torch.full((1, keys, 64), 100, dtype=torch.int8)
    k = torch.randint(-1, 2, (1, keys, 64), generator=g, dtype=torch.int8)
    v = torch.randint(1, 128, (1, keys, 64), generator=g, dtype=torch.int8)
    k[0, 0], v[0, 0] = 100, 0
    scale = torch.tensor([(gap * 8 * np.log(2) / 640000) ** 0.5], dtype=torch.float32)
    qd, kd, vd = (t.double() * scale.double() for t in (q, k, v))
    want = torch.softmax(qd @ kd.transpose(1, 2) / 8.0, -1) @ vd
    got = K.attention(torch.cat([q, k, v], -1).cuda(), 1, qkv_scale=scale.cuda()).cpu().double()
    assert ((got - want) / want).abs().max().item() <= (2.5 * gap + 170) * 2.0 ** -24


def test_attention_takes_an_int8_projection_with_its_scale_only(K):
    codes = torch.zeros((1, 2, 192), dtype=torch.int8, device="cuda")
    for args in ((codes, 1), (codes, 1, None, torch.ones(2, device="cuda")), (codes, 1, None, torch.ones(1)),
                 (codes.float(), 1, None, 1.0)):
        with pytest.raises((TypeError, ValueError)):
            K.attention(*args)


@pytest.mark.parametrize("rows,cols", [(1, 4), (5, 252), (3, 260), (9, 768), (1026, 1000), (7, 1028), (2, 2048)])
def test_layer_norm_with_and_without_its_quantize(K, rows, cols):
    g = torch.Generator().manual_seed(cols)
    x = torch.randn(rows, cols, generator=g) * 3 + 1
    gamma, beta = torch.randn(cols, generator=g), torch.randn(cols, generator=g)
    want = torch.nn.functional.layer_norm(x.double(), (cols,), gamma.double(), beta.double(), 1e-12)
    y = K.layer_norm(x.cuda(), gamma.cuda(), beta.cuda(), 1e-12)
    torch.testing.assert_close(y.cpu().double(), want, rtol=1e-5, atol=2e-5)
    scale = torch.full((1,), 0.03, device="cuda")
    y2, q = K.layer_norm(x.cuda(), gamma.cuda(), beta.cuda(), 1e-12, scale)
    assert torch.equal(y2, y)
    assert torch.equal(q, K.quantize(y, scale, torch.zeros(1, dtype=torch.int32, device="cuda")))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("m,k,n", [(1, 16, 1), (3, 17, 33), (16, 63, 40), (17, 65, 31), (32, 2047, 129), (33, 79, 65), (40, 1001, 300),
                                   (100, 3009, 96), (129, 130, 700), (600, 2057, 130)])
def test_weight_only_qgemm_rows_of_any_length_and_alignment(K, dtype, m, k, n):
    """Row lengths that are multiples of nothing, and 16-byte lengths at odd bases, on either side
    of the k tiles, of the row limits and of the tile sizes; one launch and split over k."""
    rng = np.random.default_rng(m + k + n)
    for signed in (False, True):
        x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, signed)
        for ws in (True, False):
            got = K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), dev(bias), workspace=ws)
            _weight_only_check(got, x, w, scale, zp, bias, dtype)
        got = K.weight_only_qgemm(dev(x), dev(np.ascontiguousarray(w.T)), dev(scale), dev(zp), None, tp_b=False)
        _weight_only_check(got, x, w, scale, zp, None, dtype)
    x, w, scale, zp, bias = _weight_only_case(rng, m, (k + 15) // 16 * 16, n, dtype, False)
    xb = torch.empty(x.size + 1, dtype=dtype, device="cuda")[1:].view(x.shape).copy_(dev(x))
    wb = torch.empty(w.size + 3, dtype=torch.uint8, device="cuda")[3:].view(w.shape).copy_(dev(w))
    _weight_only_check(K.weight_only_qgemm(xb, wb, dev(scale), dev(zp), dev(bias)), x, w, scale, zp, bias, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n", [1, 47, 4097, 8200, 12300])
@pytest.mark.parametrize("m", [2, 16, 17, 32])
def test_weight_only_qgemm_few_rows_at_every_workgroup_width(K, dtype, m, n):
    """16, 32, 48 and 64 channels per workgroup (N up to 4096, 8192, 12288, 16384 on 256 compute units),
    the last one partly filled; k of part of a unit, of an uneven number of units per wave, and past a
    whole round of the waves; rows off 16 bytes."""
    rng = np.random.default_rng(m + n)
    for k in (16, 1040, 2112, 1043):
        x, w, scale, zp, bias = _weight_only_case(rng, m, k, n, dtype, k == 1040)
        _weight_only_check(K.weight_only_qgemm(dev(x), dev(w), dev(scale), dev(zp), dev(bias)), x, w, scale,
                           zp, bias, dtype)


@pytest.mark.parametrize("m,k,n", [(1, 64, 3), (1, 64, 4), (33, 128, 37), (65, 64, 68), (130, 768, 66), (257, 3072, 132),
                                   (1000, 256, 256)])
def test_residual_behind_f32_results_at_the_edges_of_the_fragments(K, m, k, n):
    """Rows and columns of a fragment past the result, N below and off a group of four, k in one and
    in several wave groups: the bits of the dequantized result and a separate addition."""
    g = torch.Generator().manual_seed(m + n)
    a = torch.randint(-128, 128, (m, k), generator=g, dtype=torch.int8).cuda()
    w = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8).cuda()
    sx, so = torch.tensor([0.02]).cuda(), torch.tensor([0.05 * k ** 0.5]).cuda()
    sw = (torch.rand(n, generator=g) * 0.01 + 0.01).cuda()
    run = lambda **kw: K.qgemm(a, w, K.EPI_REQUANT_CPU_DEQUANT_F32, sx=sx, sw=sw, so=so, **kw)  # noqa: E731
    plain = run()
    r = torch.randn(m, n, generator=g).cuda()
    assert torch.equal(run(post=K.make_postops(residual=r)), plain + r)
    q = torch.randint(-128, 128, (m, n), generator=g, dtype=torch.int8).cuda()
    assert torch.equal(run(post=K.make_postops(residual=q, residual_scale=sx)), plain + q.float() * sx)


def test_operators_on_tensors_without_storage_or_rows_raise(K):
    """What cannot be launched on raises an ordinary exception before anything is launched: a result
    of rank 0 where rows are written, a tensor under torch.vmap, a sparse bias."""
    i8 = torch.zeros((4, 64), dtype=torch.int8, device="cuda")
    f32 = torch.zeros((4, 64), device="cuda")
    one, zero = torch.ones(1, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    sc = dict(sx=one, sw=one, so=one)
    table = torch.zeros(256, dtype=torch.int8, device="cuda")
    refusals = (IndexError, RuntimeError, NotImplementedError)

    def rank0(dtype):
        return torch.zeros((), dtype=dtype, device="cuda")

    for call in (lambda: K.qgemm(i8, i8, K.EPI_ACC_S32, out=rank0(torch.int32)),
                 lambda: K.qlinear_f32(f32, i8, K.EPI_REQUANT_CPU, out=rank0(torch.int8), **sc),
                 lambda: K.weight_only_qgemm(f32, i8, f32[:, 0], out=rank0(torch.float32)),
                 lambda: K.qgemm(i8, i8, K.EPI_REQUANT_CPU, bias=f32[0, :4].to_sparse(), **sc)):
        with pytest.raises(refusals):
            call()
    batch8, batch32 = i8.reshape(2, 2, 64), f32.reshape(2, 2, 64)
    lo, hi = one.clone(), one.clone()
    for fn, arg in ((lambda t: K.quantize(t, one, zero), batch32), (lambda t: K.fake_quant(t, one, zero), batch32),
                    (lambda t: K.dequantize(t, one, zero), batch8), (lambda t: K.lut8(t, table), batch8),
                    (lambda t: K.minmax(t, lo, hi)[0], batch32),
                    (lambda t: K.observe(t, lo, hi, True, -128, 127, fake_quant=True)[3], batch32),
                    (lambda t: K.qgemm(t, i8, K.EPI_ACC_S32), batch8),
                    (lambda t: K.qlinear_f32(t, i8, K.EPI_REQUANT_CPU, **sc), batch32),
                    (lambda t: K.weight_only_qgemm(t, i8, f32[:, 0]), batch32),
                    (lambda t: K.layer_norm(t, f32[0], f32[0]), batch32),
                    (lambda t: K.attention(t, 1), torch.zeros((2, 1, 2, 192), device="cuda")),
                    (lambda t: K.qconv2d(t, i8.reshape(4, 1, 1, 64), [0] * 4, list(O.NHWC_OHWI_METADATA) + [1] * 5,
                                         [1, 1, 2, 4], K.EPI_ACC_S32), batch8.reshape(2, 1, 1, 2, 64))):
        with pytest.raises(refusals):
            torch.vmap(fn)(arg)
    assert torch.equal(K.lut8(i8, table), i8)       # (and the next call works)


@pytest.mark.parametrize("s", [17, 64, 65, 130, 200])
def test_attention_with_infinite_scores_and_values(K, s):
    """Scores of -inf for the first keys (all of the first 64 where there are more), for every key,
    and of +inf; infinite values in the last token, next to the rows past the sequence: the f64
    result, NaN where that is NaN."""
    g = torch.Generator().manual_seed(s)
    qkv = torch.randn(3, s, 3 * 64, generator=g)
    q, k, v = qkv[..., :64], qkv[..., 64:128], qkv[..., 128:]
    q[..., 0] = q[..., 0].abs() + 0.5
    q[0, 1, 0] = -1.0                                # +inf scores: no probability is defined
    k[0, :min(64, s - 1), 0] = -float("inf")         # (the keys behind them decide)
    k[1, :, 0] = -float("inf")
    v[2, -1, 3], v[2, -1, 40] = float("inf"), -float("inf")
    qd, kd, vd = q.double(), k.double(), v.double()
    want = torch.softmax(qd @ kd.transpose(1, 2) / 8.0, -1) @ vd
    assert not want[0, 0].isnan().any() and want[0, 1].isnan().all() and want[1].isnan().all()
    assert (want[2, :, 3] == float("inf")).all() and (want[2, :, 40] == -float("inf")).all()
    got = K.attention(qkv.cuda(), 1)
    torch.testing.assert_close(got.cpu().double(), want, rtol=1e-5, atol=1e-5, equal_nan=True)
    scale = torch.full((1,), 0.02, device="cuda")
    got_q = K.attention(qkv.cuda(), 1, scale)
    assert torch.equal(got_q, K.quantize(got, scale, torch.zeros(1, dtype=torch.int32, device="cuda")))
    assert (got_q[2, :, 3] == 127).all() and (got_q[2, :, 40] == -128).all()


@pytest.mark.parametrize("m,n,k,tp_a,tp_b", [(300, 260, 784, 0, 0), (300, 260, 272, 1, 0), (129, 70, 1041, 1, 1),
                                             (1000, 768, 777, 0, 1), (17, 33, 16, 0, 0)])
@pytest.mark.parametrize("zx,zw", [(0, 0), (-11, 0), (5, -3)])
def test_qgemm_scratch_for_rows_of_k_rounded_up_to_16(K, m, n, k, tp_a, tp_b, zx, zw):
    """Scratch counted with rows of K rounded up to 16 bytes, less than dq8_qgemm_workspace_bytes
    asks for, is enough, with and without room for the zero-point corrections; nothing behind it
    is written."""
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-128, 128, (k, m) if tp_a else (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k) if tp_b else (k, n), dtype=np.int8)
    want = ((a.T if tp_a else a).astype(np.int64) - zx) @ ((w if tp_b else w.T).astype(np.int64) - zw).T
    up = lambda v: (v + 255) // 256 * 256      # noqa: E731
    k16 = (k + 15) // 16 * 16
    rows = (up(m * k16) if tp_a or k % 16 else 0) + (up(n * k16) if not tp_b or k % 16 else 0)
    L, da, dw = K._lib.lib(), dev(a), dev(w)
    for size in {rows, rows + (up(4 * n) + up(4 * m) if zx or zw else 0)}:
        ws = torch.full((size + 256,), 77, dtype=torch.uint8, device="cuda")
        out = torch.empty((m, n), dtype=torch.int32, device="cuda")
        st = L.dq8_qgemm(K._ptr(da), da.stride(0), K._ptr(dw), dw.stride(0), K._ptr(out), n, m, n, k, tp_a, tp_b,
                         K.EPI_ACC_S32, None, 0, None, 0, None, 0, None, 0, zx, zw, 0, K._ptr(ws), size, K._stream())
        K._lib.check(st, "dq8_qgemm")
        np.testing.assert_array_equal(host(out), want)
        assert (ws[size:] == 77).all()


def test_bounds_and_scales_in_every_form_python_has_for_them(K):
    """quantize's bounds as floats, a GEMM's scales as a number, list, numpy array or tensor of any
    float type: the results of integers and flat f32 device tensors."""
    rng = np.random.default_rng(5)
    x = dev(rng.standard_normal((6, 64)).astype(np.float32))
    one, zero = torch.full((1,), 0.05, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    q = K.quantize(x, one, zero, qmin=-7, qmax=100)
    for lo, hi in ((-7.0, 100.0), (np.float32(-7), np.int64(100)), (np.float64(-7.9), 100.5)):
        assert torch.equal(K.quantize(x, one, zero, qmin=lo, qmax=hi), q)
    w = dev(rng.integers(-128, 128, (5, 64), dtype=np.int8))
    s = rng.uniform(0.01, 0.02, 5).astype(np.float32)
    sx, so = np.float32(0.05), np.float32(0.3)
    want = K.qgemm(q, w, K.EPI_REQUANT_CPU, sx=dev(sx.reshape(1)), sw=dev(s), so=dev(so.reshape(1)))
    assert want.abs().max() > 0
    for a, b, c in ((float(sx), s.tolist(), float(so)), (sx, s, so), ([float(sx)], s.astype(np.float64), so.reshape(1, 1)),
                    ((float(sx),), tuple(s.tolist()), so),
                    (dev(sx.reshape(1)), dev(s).double().reshape(5, 1), dev(np.stack([so, so]))[:1])):
        assert torch.equal(K.qgemm(q, w, K.EPI_REQUANT_CPU, sx=a, sw=b, so=c), want)
    want = K.qlinear_f32(x, w, K.EPI_REQUANT_CPU, sx=dev(sx.reshape(1)), sw=dev(s), so=dev(so.reshape(1)))
    assert torch.equal(K.qlinear_f32(x, w, K.EPI_REQUANT_CPU, sx=float(sx), sw=s.tolist(), so=so), want)
    for bad in ("0.05", {}, object()):
        with pytest.raises((TypeError, ValueError, RuntimeError)):
            K.qgemm(q, w, K.EPI_REQUANT_CPU, sx=bad, sw=s.tolist(), so=so)


def test_results_into_lazy_copies_leave_the_original_alone(K):
    """A result tensor or a running state that shares its memory with another one until it is
    written (copy on write)."""
    f32 = torch.randn((4, 64), device="cuda")
    i8 = torch.randint(-128, 128, (4, 64), dtype=torch.int8, device="cuda")
    one, zero = torch.full((1,), 0.05, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    table = torch.arange(256, device="cuda").to(torch.uint8).view(torch.int8)
    md = list(O.NHWC_OHWI_METADATA) + [1] * 5
    for run, shape, dtype in ((lambda o: K.quantize(f32, one, zero, out=o), (4, 64), torch.int8),
                              (lambda o: K.dequantize(i8, one, zero, out=o), (4, 64), torch.float32),
                              (lambda o: K.fake_quant(f32, one, zero, out=o), (4, 64), torch.float32),
                              (lambda o: K.lut8(i8, table, out=o), (4, 64), torch.int8),
                              (lambda o: K.qgemm(i8, i8, K.EPI_ACC_S32, out=o), (4, 4), torch.int32),
                              (lambda o: K.weight_only_qgemm(f32, i8, one.expand(4), out=o), (4, 4), torch.float32),
                              (lambda o: K.qlinear_f32(f32, i8, K.EPI_DEQUANT_F32, one, one, out=o), (4, 4), torch.float32),
                              (lambda o: K.qconv2d(i8.reshape(1, 1, 4, 64), i8.reshape(4, 1, 1, 64), [0] * 4, md,
                                                   [1, 1, 4, 4], K.EPI_ACC_S32, out=o), (1, 1, 4, 4), torch.int32),
                              (lambda o: K.minmax(f32, o, one.clone()), (1,), torch.float32),
                              (lambda o: K.observe(f32, o, one.clone(), True, -128, 127), (1,), torch.float32)):
        original = torch.full(shape, 99, dtype=dtype, device="cuda")
        copy = torch._lazy_clone(original)
        run(copy)
        assert (original == 99).all()
        assert not torch.equal(copy, original)


def _fused_forms_equal_the_separate_operators(K, a, w, zx, rng):
    """Everything dq8_qgemm fuses behind a product with an input zero point, into results of their
    own and into rows that begin at any byte, against the scalar kernel and the operators by
    themselves."""
    (m, k), n, gen = a.shape, w.shape[0], 0
    so = np.float32(0.02 * 0.025 * 74.0 * 74.0 * np.sqrt(k) / 40.0)
    dso, sr, s2 = (dev(np.array([v], np.float32)) for v in (so, so * 0.7, so * 1.4))
    zi = lambda v: torch.full((1,), v, dtype=torch.int32, device="cuda")  # noqa: E731
    sc = dict(sx=dev(np.array([0.02], np.float32)), so=dso, sw=dev(rng.uniform(0.001, 0.05, n).astype(np.float32)), zx=zx)
    bias = dev((rng.standard_normal(n) * 20 * so).astype(np.float32))
    b32 = dev(rng.integers(-20000, 20000, n).astype(np.int32))
    q = K.qgemm(a, w, K.EPI_REQUANT_CPU, bias=bias, zo=2, variant=gen, **sc)
    y = K.dequantize(q, dso, zi(2))
    wide8, wide32 = torch.empty((m, n + 3), dtype=torch.int8, device="cuda"), torch.empty((m, n + 1), device="cuda")
    res8 = dev(rng.integers(-128, 128, (m, n + 5), dtype=np.int8))
    res32 = dev((rng.standard_normal((m, n + 3)) * 40 * so).astype(np.float32))
    outs8, outs32 = (None, wide8[:, 1:n + 1]), (None, wide32[:, 1:])
    table = dev(rng.integers(-128, 128, 256, dtype=np.int8))
    clamp = dev(np.clip(np.arange(256).astype(np.uint8).view(np.int8), 0, 100).astype(np.int8))
    for t in (table, clamp):
        for out in outs8:
            got = K.qgemm(a, w, K.EPI_REQUANT_CPU, bias=bias, zo=2, out=out, post=K.make_postops(table=t), **sc)
            assert torch.equal(got, K.lut8(q, t))
    for r8 in (res8[:, :n].contiguous(), res8[:, 2:n + 2]):
        t = y + K.dequantize(r8.contiguous(), sr, zi(-4))
        relu = torch.where(t < 0, torch.zeros_like(t), t)
        for out in outs8:
            got = K.qgemm(a, w, K.EPI_REQUANT_CPU, bias=bias, zo=2, out=out, post=K.make_postops(
                residual=r8, residual_scale=sr, residual_zp=-4, relu=True, out_scale=s2, out_zp=-9), **sc)
            assert torch.equal(got, K.quantize(relu, s2, zi(-9)))
        for out in outs32:
            got = K.qgemm(a, w, K.EPI_REQUANT_CPU_DEQUANT_F32, bias=bias, zo=2, out=out,
                          post=K.make_postops(residual=r8, residual_scale=sr, residual_zp=-4), **sc)
            assert torch.equal(got.contiguous().view(torch.int32), t.view(torch.int32))
    for r32 in (res32[:, :n].contiguous(), res32[:, 1:n + 1]):
        t = y + r32
        for out in outs32:
            got = K.qgemm(a, w, K.EPI_REQUANT_CPU_DEQUANT_F32, bias=bias, zo=2, out=out,
                          post=K.make_postops(residual=r32), **sc)
            assert torch.equal(got.contiguous().view(torch.int32), t.view(torch.int32))
        for out in outs8:
            got = K.qgemm(a, w, K.EPI_REQUANT_CPU, bias=bias, zo=2, out=out,
                          post=K.make_postops(residual=r32, out_scale=s2), **sc)
            assert torch.equal(got, K.quantize(t, s2, zi(0)))
    fix = K.qgemm(a, w, K.EPI_REQUANT_FIXEDPOINT, bias=b32, zo=-3, variant=gen, **sc)
    for out in outs8:
        assert torch.equal(K.qgemm(a, w, K.EPI_REQUANT_FIXEDPOINT, bias=b32, zo=-3, out=out, **sc), fix)
        got = K.qgemm(a, w, K.EPI_REQUANT_FIXEDPOINT, bias=b32, zo=-3, out=out, post=K.make_postops(table=table), **sc)
        assert torch.equal(got, K.lut8(fix, table))
    assert q.unique().numel() > 20


# shapes of every tile that sums the zero point up in its k loop, and of the small-M kernel
ZP_TILES = [((300, 261, 96), "pipe_64x64x128"), ((1100, 770, 2064), "pipe_64x64x128_k2"),
            ((256, 512, 8192), "pipe_64x64x128_k4"), ((2048, 2048, 4096), "pipe_128x128x128"),
            ((4097, 768, 272), "pipe_128x128x128_w8"), ((4096, 4096, 256), "pipe_256x256x128_w8"),
            ((4000, 3070, 256), "pipe_256x192x128_w8"), ((33, 257, 80), "skinny_16")]


@pytest.mark.parametrize("shape,kernel", ZP_TILES, ids=[t[1] for t in ZP_TILES])
def test_fused_operators_behind_a_zero_point_in_the_k_loop(K, shape, kernel):
    m, n, k = shape
    assert K._lib.lib().dq8_qgemm_kernel_name(m, n, k, 1).decode() == kernel
    rng = np.random.default_rng(m + n + k)
    a, w = dev(rng.integers(-128, 128, (m, k), dtype=np.int8)), dev(rng.integers(-128, 128, (n, k), dtype=np.int8))
    for zx in (-11, 100):
        _fused_forms_equal_the_separate_operators(K, a, w, zx, rng)


# and of the tiles whose k tiles are dealt out over the waves: fewer k tiles than waves, one more than whole
# rounds of them, rows and channels that end inside a tile
WAVE_TILES = [((330, 272, 96), "wave_32x32_w4"), ((410, 560, 528), "wave_32x32_w4"), ((343, 512, 2064), "wave_32x32_w8"),
              ((335, 1168, 320), "wave_32x64_w4"), ((519, 848, 1040), "wave_32x64_w4"), ((1100, 784, 2064), "wave_64x64_w4"),
              ((1300, 1008, 2064), "wave_96x64_w4"), ((260, 130, 1040), "wave_32x32_w8"), ((519, 847, 1040), "wave_32x64_w4"),
              ((1021, 1001, 2320), "wave_64x64_w4"), ((1250, 1006, 2576), "wave_96x64_w4")]


@pytest.mark.parametrize("shape,kernel", WAVE_TILES, ids=["%s-%d" % (t[1], t[0][2]) for t in WAVE_TILES])
def test_fused_operators_behind_k_tiles_dealt_out_over_the_waves(K, shape, kernel):
    m, n, k = shape
    assert K._lib.lib().dq8_qgemm_kernel_name(m, n, k, 1).decode() == kernel
    rng = np.random.default_rng(m + n + k)
    a, w = dev(rng.integers(-128, 128, (m, k), dtype=np.int8)), dev(rng.integers(-128, 128, (n, k), dtype=np.int8))
    for zx in (0, -11):
        _fused_forms_equal_the_separate_operators(K, a, w, zx, rng)


@pytest.mark.parametrize("shape,kernel", [WAVE_TILES[i] for i in (1, 2, 3, 5, 6, 8, 9, 10)],
                         ids=["%s-%d" % (t[1], t[0][2]) for t in (WAVE_TILES[i] for i in (1, 2, 3, 5, 6, 8, 9, 10))])
def test_zero_point_of_the_weights_behind_k_tiles_dealt_out_over_the_waves(K, shape, kernel):
    """The row sums of both operands, added by the owner of each fragment -- rows and channels of every fragment of
    the tile, and those past the edges."""
    m, n, k = shape
    rng = np.random.default_rng(m + n + k)
    a, w = dev(rng.integers(-128, 128, (m, k), dtype=np.int8)), dev(rng.integers(-128, 128, (n, k), dtype=np.int8))
    sc = dict(sx=dev(np.array([0.02], np.float32)), sw=dev(rng.uniform(0.001, 0.05, n).astype(np.float32)),
              so=dev(np.array([3.0], np.float32)), bias=dev(rng.standard_normal(n).astype(np.float32)))
    assert K._lib.lib().dq8_qgemm_kernel_name(m, n, k, 1).decode() == kernel
    for epi in (K.EPI_REQUANT_CPU, K.EPI_REQUANT_GPU, K.EPI_ACC_S32, K.EPI_REQUANT_CPU_DEQUANT_F32):
        kw = {} if epi == K.EPI_ACC_S32 else sc
        for zx, zw in ((0, 5), (-11, -7)):
            want = K.qgemm(a, w, epi, variant=0, zx=zx, zw=zw, **kw)
            assert torch.equal(K.qgemm(a, w, epi, zx=zx, zw=zw, **kw), want), (epi, zx, zw)


@pytest.mark.parametrize("nb,h,w_,ci,co,kk,stride,pad,dil", [
    (1, 7, 7, 16, 32, 1, 1, 0, 1), (2, 9, 11, 48, 72, 3, 1, 1, 1), (3, 7, 7, 512, 48, 3, 1, 1, 1),
    (1, 13, 10, 80, 33, 3, 2, 1, 1), (2, 12, 9, 32, 64, 5, 1, 2, 1), (1, 15, 15, 208, 96, 3, 1, 2, 2),
    (5, 14, 14, 256, 65, 1, 2, 0, 1), (2, 20, 6, 144, 40, 2, 3, 1, 1)])
def test_convolutions_on_k_tiles_dealt_out_over_the_waves(K, nb, h, w_, ci, co, kk, stride, pad, dil):
    """Forced, against the generic kernel: taps in the padding, a k tile that begins inside a tap (the tap of a
    wave's next tile is had by additions, several taps and a row of the filter on), images that end inside a
    tile; and as the library runs them (a strided 1 x 1 filter as a GEMM over its pixels)."""
    rng = np.random.default_rng(h * w_ + ci + co + kk)
    x = dev(rng.integers(-128, 128, (nb, h, w_, ci), dtype=np.int8))
    wt = dev(rng.integers(-128, 128, (co, kk, kk, ci), dtype=np.int8))
    ho = (h + 2 * pad - dil * (kk - 1) - 1) // stride + 1
    wo = (w_ + 2 * pad - dil * (kk - 1) - 1) // stride + 1
    md = list(O.NHWC_OHWI_METADATA) + [stride, stride, dil, dil, 1]
    sc = dict(sx=dev(np.array([0.02], np.float32)), sw=dev(rng.uniform(0.001, 0.05, co).astype(np.float32)),
              so=dev(np.array([0.5], np.float32)), bias=dev(rng.standard_normal(co).astype(np.float32)))
    waves = [i for i, nm in enumerate(K.variant_names()) if nm.startswith("wave_")]
    assert len(waves) == 5 and K.variant_names()[waves.pop()] == "wave_96x64_w4"   # (products only)
    for epi in (K.EPI_ACC_S32, K.EPI_REQUANT_CPU, K.EPI_REQUANT_CPU_DEQUANT_F32):
        kw = {} if epi == K.EPI_ACC_S32 else sc
        want = K.qconv2d(x, wt, [pad] * 4, md, [nb, ho, wo, co], epi, variant=0, **kw)
        for v in waves + [-1]:
            got = K.qconv2d(x, wt, [pad] * 4, md, [nb, ho, wo, co], epi, variant=v, **kw)
            assert torch.equal(got, want), (v, epi)


WORDS, SMALL_M, REGISTERS = 1, 2, 3


def _rows_kernel(a, w, out_bytes):
    """(form, kernel) that dq8_qgemm plans for these operands' rows off 16 bytes."""
    import ctypes as C
    import bladedisc_amd._lib as _lib
    form = C.c_int()
    name = _lib.hooks().dq8_qgemm_rows_kernel(a.shape[0], w.shape[0], a.shape[1], a.stride(0), w.stride(0), a.data_ptr() % 16,
                                         w.data_ptr() % 16, 0, out_bytes, C.byref(form))
    return form.value, name.decode()


# the same for operand rows of any length and alignment
RAGGED_TILES = [((300, 261, 90), "pipe_64x64x128"), ((260, 130, 1001), "pipe_64x64x128"),
                ((1100, 770, 2058), "pipe_64x64x128_k2"), ((320, 513, 8206), "pipe_64x64x128_k4"),
                ((33, 257, 79), "skinny_16")]


@pytest.mark.parametrize("shape,kernel", RAGGED_TILES, ids=["%s-%d" % (t[1], t[0][2]) for t in RAGGED_TILES])
def test_fused_operators_behind_rows_of_any_length(K, shape, kernel):
    m, n, k = shape
    rng = np.random.default_rng(m + n + k)
    wide_a = dev(rng.integers(-128, 128, (m, (k + 11) // 4 * 4), dtype=np.int8))
    wide_w = dev(rng.integers(-128, 128, (n, (k + 15) // 4 * 4), dtype=np.int8))
    # (rows on four bytes at any k, at odd bytes up to 2048 of k: what the tiles take as they are)
    forms = [(wide_a[:, 4:4 + k], wide_w[:, 8:8 + k])] + \
        ([(wide_a[:, :k].contiguous(), wide_w[:, :k].contiguous()), (wide_a[:, 3:3 + k], wide_w[:, 1:1 + k])]
         if k <= 2048 else [])
    for a, w in forms:
        assert _rows_kernel(a, w, 1) == (SMALL_M if kernel == "skinny_16" else REGISTERS, kernel)
        for zx in (0, -11):
            _fused_forms_equal_the_separate_operators(K, a, w, zx, rng)


# operand rows on four bytes: (m, n, k) and the tile that an int8 result gets
WORD_TILES = [((400, 256, 500), "wave_32x32_w8"), ((300, 257, 1036), "wave_32x32_w8"), ((335, 1152, 324), "wave_32x64_w4"),
              ((1023, 897, 4108), "wave_64x64_w4"), ((777, 1501, 1000), "pipe_64x64x128"), ((640, 513, 124), "pipe_64x64x128"),
              ((513, 1023, 2052), "pipe_64x64x128_k2"), ((4097, 1281, 264), "pipe_128x128x128_w8"),
              ((4090, 3500, 396), "pipe_256x256x128_w8"), ((1300, 1024, 2500), "pipe_64x64x128"), ((777, 1501, 1024), "pipe_64x64x128"),
              # the small-M kernel chosen and not taken
              ((283, 618, 2628), "wave_32x32_w8"), ((130, 1306, 1416), "wave_32x32_w8"), ((32, 8640, 2052), "wave_32x64_w4")]


@pytest.mark.parametrize("shape,kernel", WORD_TILES, ids=["%s-%d" % (t[1], t[0][2]) for t in WORD_TILES])
def test_qgemm_on_rows_that_begin_on_four_bytes(K, shape, kernel):
    """Rows of whole words, contiguous and out of wider rows whose other bytes are not zero: every place of the
    rows' end in a k tile's steps, a wave's half and a chunk.  Sums of whole numbers: equal bits."""
    m, n, k = shape
    rng = np.random.default_rng(m + n + k)
    wide_a = dev(rng.integers(-128, 128, (m, k + 12), dtype=np.int8))
    wide_w = dev(rng.integers(-128, 128, (n, k + 20), dtype=np.int8))
    sc = dict(sx=dev(np.array([0.02], np.float32)), sw=dev(rng.uniform(0.001, 0.05, n).astype(np.float32)),
              so=dev(np.array([3.0], np.float32)), bias=dev(rng.standard_normal(n).astype(np.float32)))
    last = [k] if k > 1500 else [k, k - 4, k - 8, k - 12, k - 20, k - 36]
    for kk in last:
        for a, w in ((wide_a[:, :kk].contiguous(), wide_w[:, :kk].contiguous()),
                     (wide_a[:, 4:4 + kk], wide_w[:, 8:8 + kk])):
            form, name = _rows_kernel(a, w, 1)       # (of what is not aligned after all another kernel runs)
            assert form == _rows_kernel(a, w, 4)[0] == WORDS and (kk != k or name == kernel)
            for zx in (0, -11):
                acc = K.qgemm(a, w, K.EPI_ACC_S32, variant=0, zx=zx)
                assert torch.equal(K.qgemm(a, w, K.EPI_ACC_S32, zx=zx), acc)
                for epi in (K.EPI_REQUANT_CPU, K.EPI_REQUANT_GPU, K.EPI_REQUANT_CPU_DEQUANT_F32):
                    want = K.qgemm(a, w, epi, variant=0, zx=zx, **sc)
                    assert torch.equal(K.qgemm(a, w, epi, zx=zx, **sc), want), (kk, zx, epi)


@pytest.mark.parametrize("shape,kernel", [
    ((335, 1168, 324), "wave_32x64_w4"), ((300, 261, 1036), "wave_32x32_w8"), ((1023, 897, 2316), "wave_64x64_w4"),
    ((777, 1501, 516), "pipe_64x64x128"), ((320, 513, 8204), "pipe_64x64x128_k2"), ((4097, 1281, 268), "pipe_128x128x128_w8"),
    ((4090, 3500, 264), "pipe_256x256x128_w8")])
def test_fused_operators_behind_rows_of_whole_words(K, shape, kernel):
    """Every tile that has a form for such rows."""
    m, n, k = shape
    rng = np.random.default_rng(m + n + k)
    a = dev(rng.integers(-128, 128, (m, k + 12), dtype=np.int8))[:, 4:4 + k]
    w = dev(rng.integers(-128, 128, (n, k + 20), dtype=np.int8))[:, 8:8 + k]
    assert _rows_kernel(a, w, 1) == (WORDS, kernel)
    for zx in (0, -11):
        _fused_forms_equal_the_separate_operators(K, a, w, zx, rng)


@pytest.mark.parametrize("rows,nch", [(4, 3), (5, 37), (1023, 255), (7, 256), (64, 257), (33, 511), (9, 1025),
                                      (4, 3073), (517, 1537), (1021, 1), (1723, 2501)])
@pytest.mark.parametrize("xt,qt", [(torch.float32, torch.uint8), (torch.float16, torch.int8),
                                   (torch.float32, torch.int16), (torch.float16, torch.int16),
                                   (torch.float32, torch.int32)])
def test_quantize_by_channel_and_by_sweep_any_type(K, rows, nch, xt, qt):
    """Per channel of the last axis and per tensor, at the edges of the four-row groups, of a workgroup's
    1024, 2048 or 4096 elements and of the choice between the two kernels; with values whose quotients are
    not finite and, in a second pass, scales that no reciprocal is used for.  Every step is one rounded
    binary32 operation: equal bits."""
    rng = np.random.default_rng(rows * 4096 + nch)
    info = torch.iinfo(qt)
    lo, hi = np.float32(info.min), np.float32(info.max)
    x = (rng.standard_normal((rows, nch)) * 8).astype(np.float32)
    x.reshape(-1)[rng.integers(0, x.size, 9)] = [np.nan, np.inf, -np.inf, 0.0, -0.0, 6e4, -6e4, 0.5, np.nan]
    x = torch.from_numpy(x).to(xt)
    for wild in (False, True):
        scale = (rng.random(nch) * 0.05 + 0.01).astype(np.float32)
        if wild:
            scale[rng.integers(0, nch, 3)] = [1e-30, 1e30, 0.0]
        zp = rng.integers(-3 if info.min < 0 else 0, 4, nch).astype(np.int32)
        for axis in (1, None):
            if axis is None and wild:
                continue
            s, z = (scale, zp) if axis == 1 and nch > 1 else (scale[:1], zp[:1])
            ds, dz = torch.from_numpy(s).cuda(), torch.from_numpy(z).cuda()
            q = K.quantize(x.cuda(), ds, dz, axis=axis, qmin=info.min, qmax=info.max, dtype=qt)
            with np.errstate(all="ignore"):
                t = np.rint(x.float().numpy() / s + z.astype(np.float32))
            want = np.clip(np.fmin(np.fmax(t, lo), hi).astype(np.float64), info.min, info.max).astype(np.int64)
            assert np.array_equal(q.cpu().numpy().astype(np.int64), want)
            y = K.dequantize(q, ds, dz, axis=axis)
            with np.errstate(all="ignore"):
                back = (want.astype(np.int32) - z).astype(np.float32) * s
            assert np.array_equal(y.cpu().numpy().view(np.int32), back.view(np.int32))
            if xt == torch.float32 and qt in (torch.uint8, torch.int16):
                f = K.fake_quant(x.cuda(), ds, dz, axis=axis, qmin=info.min, qmax=info.max)
                assert np.array_equal(f.cpu().numpy(), back)


@pytest.mark.parametrize("outer,nch,inner", [(1, 400001, 4), (3, 70001, 9), (1, 1537, 1025), (2, 3, 400003),
                                             (5, 300, 1024), (1, 7, 5), (700, 3, 1021)])
@pytest.mark.parametrize("xt,qt", [(torch.float32, torch.uint8), (torch.float16, torch.int16),
                                   (torch.float32, torch.int32)])
def test_quantize_by_row_any_type(K, outer, nch, inner, xt, qt):
    """The channel on an axis that is not the last, rows of any length from four elements on: groups across
    the end of a row, several rows per workgroup, scales that no reciprocal is used for.  Equal bits."""
    rng = np.random.default_rng(nch * 16 + inner)
    info = torch.iinfo(qt)
    x = (rng.standard_normal((outer, nch, inner)) * 8).astype(np.float32)
    x.reshape(-1)[rng.integers(0, x.size, 6)] = [np.nan, np.inf, -np.inf, 0.0, 6e4, -6e4]
    x = torch.from_numpy(x).to(xt)
    s = (rng.random(nch) * 0.05 + 0.01).astype(np.float32)
    s[rng.integers(0, nch, 3)] = [1e-30, 1e30, 0.0]
    z = rng.integers(0, 4, nch).astype(np.int32)
    ds, dz = torch.from_numpy(s).cuda(), torch.from_numpy(z).cuda()
    q = K.quantize(x.cuda(), ds, dz, axis=1, qmin=info.min, qmax=info.max, dtype=qt)
    with np.errstate(all="ignore"):
        t = np.rint(x.float().numpy() / s[:, None] + z[:, None].astype(np.float32))
    want = np.clip(np.fmin(np.fmax(t, np.float32(info.min)), np.float32(info.max)).astype(np.float64),
                   info.min, info.max).astype(np.int64)
    assert np.array_equal(q.cpu().numpy().astype(np.int64), want)
    y = K.dequantize(q, ds, dz, axis=1).cpu().numpy()
    with np.errstate(all="ignore"):
        back = (want.astype(np.int32) - z[:, None]).astype(np.float32) * s[:, None]
    assert np.array_equal(y.view(np.int32), back.view(np.int32))
    if qt == torch.uint8:
        f = K.fake_quant(x.cuda(), ds, dz, axis=1, qmin=0, qmax=255).cpu().numpy()
        assert np.array_equal(f, back)


@pytest.mark.parametrize("rows,inner", [
    # per tensor: elements behind the last four; the edges of a chunk of 1024, of the sixteen chunks of eight
    # workgroups, and of the sizes that are walked in chunks
    (1, 1), (1, 3), (1, 1023), (1, 1025), (1, 8191), (1, 8193), (1, 16383), (1, 16384), (1, 16387), (1, 24577),
    (1, (1 << 25) - 1), (1, 1 << 25), (1, (1 << 25) + 5),
    # by row: rows on both sides of 2048, one and two words a thread
    (3, 4), (5, 1024), (5, 1028), (7, 2044), (7, 2048), (7, 2052), (300, 16388), (8193, 4096), (16380, 2052)])
@pytest.mark.parametrize("qt", [torch.int8, torch.uint8])
def test_quantize_and_dequantize_in_every_order_of_the_words(K, rows, inner, qt):
    """8-bit quantize and dequantize per tensor and by row, whose workgroups take the words in an order of
    their own: every element once, nothing behind the last.  Each step is one rounded binary32 operation:
    equal bits."""
    torch.manual_seed(inner)
    info = torch.iinfo(qt)
    n = rows * inner
    scale = torch.rand(rows, device="cuda") * 0.05 + 0.01
    zp = torch.randint(0, 4, (rows,), dtype=torch.int32, device="cuda")
    axis = 0 if rows > 1 else None
    x = torch.randn((rows, inner), device="cuda")
    buf = torch.full((n + 64,), 77, dtype=qt, device="cuda")
    q = K.quantize(x, scale, zp, axis=axis, qmin=info.min, qmax=info.max, dtype=qt, out=buf[:n].view(rows, inner))
    want = torch.clamp(torch.round(x / scale[:, None] + zp[:, None]), info.min, info.max).to(torch.int32)
    assert torch.equal(q.to(torch.int32), want) and bool((buf[n:] == 77).all())
    back = torch.full((n + 64,), 7.0, device="cuda")
    y = K.dequantize(q, scale, zp, axis=axis, out=back[:n].view(rows, inner))
    assert torch.equal(y, (want - zp[:, None]).float() * scale[:, None]) and bool((back[n:] == 7).all())
