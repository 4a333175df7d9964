// The f32 operators between the quantized linears of a transformer encoder layer, each with the
// quantize that follows it in the same pass: softmax(q k^T / sqrt(d)) v, and layer normalisation.
#include "dq8_common.h"
#include "disc_q8.h"
#include "q8_elementwise.h"

#pragma clang fp contract(off)

namespace dq8 {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

// int8 of four values, dq8_quantize's bits (zero point 0, half to even)
__device__ __forceinline__ uint32_t quantize4(const v4f& v, float s, float y, bool fast) {
  using namespace elementwise;
  const float4 x = make_float4(v[0], v[1], v[2], v[3]);
  if (fast) return quant4_pack_rne(div4_by_constant(x, s, y));
  return pack4(quant_one<1>(x.x, s, 0.f, -128.f, 127.f), quant_one<1>(x.y, s, 0.f, -128.f, 127.f),
               quant_one<1>(x.z, s, 0.f, -128.f, 127.f), quant_one<1>(x.w, s, 0.f, -128.f, 127.f));
}

// 16 consecutive channels of a token, quantized or as they are
template <bool QUANT>
__device__ __forceinline__ void store_context(const v4f (&y)[4], int64_t at, float* out, int8_t* out_q,
                                              const float* q_scale) {
  if (QUANT) {
    const float sc = q_scale[0];
    const float rcp = 1.0f / sc;
    const bool fast = elementwise::divisor_in_fast_range(sc);
    uint32_t w[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) w[v] = quantize4(y[v], sc, rcp, fast);
    *reinterpret_cast<uint4*>(out_q + at) = make_uint4(w[0], w[1], w[2], w[3]);
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) *reinterpret_cast<v4f*>(out + at + 4 * v) = y[v];
  }
}

// ------------------------------------------------------------------ attention
// Heads of 64 channels, f32 throughout, on v_mfma_f32_16x16x4_f32 (64 flops per clock and SIMD, the
// bound: 8 x 128 x 12 heads are 0.4 Gflop = 2.6 us of the chip's f32 matrix rate).  A wave takes 16
// query rows, a workgroup up to four waves (64 rows) of one head; keys and values pass through LDS
// 64 at a time, the next 64 on their way in registers meanwhile.
//  * S^T = K Q^T: the keys are the MFMA's row operand, so that a lane (r, g) = (lane % 16, lane / 16)
//    holds the scores of query r with keys 4 g .. 4 g + 3 of a 16-key tile.  The 64 channels are
//    summed in the order {s, 16 + s, 32 + s, 48 + s}, s = 0 .. 15: group g then needs channels
//    16 g .. 16 g + 15 of its row, four 16-byte reads.
//  * O^T = V^T P^T: that same lane's probabilities are, as they are, the column operand of the step
//    over keys {v, 4 + v, 8 + v, 12 + v}; nothing is exchanged between lanes.  Channel 4 i + t is
//    row i of output tile t, so that a row operand is read 16 bytes at a time and a lane ends up with
//    16 consecutive channels of its query: one 16-byte store once quantized.
//  * The softmax is the online form, a maximum and a sum per query over the four lanes that share
//    it, once per 64 keys.
// The heads of all sequences run fastest over the workgroups: those of one head then meet on one XCD
// (workgroups go to the eight in turn, and the heads are most often a multiple of eight or four), and
// its keys and values are read from memory into one L2.
// LDS rows of keys are 272 bytes apart: 16 lanes reading the same channels of 16 keys then cover all
// 64 banks.
constexpr int kHead = 64, kBlock = 64;
constexpr int kKeyPitch = kHead + 4;       // floats

template <int WAVES, bool QUANT>
__global__ void __launch_bounds__(WAVES * 64)
attention_f32_kernel(const float* __restrict__ qkv, int S, uint32_t all_heads, int heads, float scale_log2,
                     float* __restrict__ out, int8_t* __restrict__ out_q, const float* __restrict__ q_scale) {
  __shared__ __attribute__((aligned(16))) float keys[kBlock * kKeyPitch];
  __shared__ __attribute__((aligned(16))) float vals[kBlock * kHead];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const uint32_t bh = blockIdx.x % all_heads, tile = blockIdx.x / all_heads;
  const int b = (int)(bh / heads), h = (int)(bh % heads);
  const int64_t row3 = 3 * (int64_t)heads * kHead;           // floats between two tokens
  const float* base = qkv + (int64_t)b * S * row3 + h * kHead;
  const int q0 = ((int)tile * WAVES + wave) * 16;

  // the wave's queries: lane (r, g) channels 16 g .. 16 g + 15 of row r, scaled by log2(e) / sqrt(d)
  v4f q[4];
  {
    const int row = q0 + r < S ? q0 + r : S - 1;
    const v4f* p = reinterpret_cast<const v4f*>(base + row * row3 + 16 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = p[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] *= scale_log2;
  }

  // 64 keys and values: 16 lanes per row
  const int lrow = threadIdx.x >> 4, lcol = (threadIdx.x & 15) * 4;
  constexpr int step = WAVES * 4;                            // rows a pass covers
  constexpr int kPasses = (kBlock + step - 1) / step;
  v4f kreg[kPasses], vreg[kPasses];
  auto fetch = [&](int key0) {
#pragma unroll
    for (int i = 0; i < kPasses; ++i) {
      const int row = lrow + i * step;
      // (zeros past the sequence: what stands there is met by a probability of zero, and zero times a
      // copy of a token with infinite values would be a NaN)
      kreg[i] = vreg[i] = (v4f){0.f, 0.f, 0.f, 0.f};
      if (row < kBlock && key0 + row < S) {
        const float* p = base + (key0 + row) * row3 + (int64_t)heads * kHead + lcol;
        kreg[i] = *reinterpret_cast<const v4f*>(p);
        vreg[i] = *reinterpret_cast<const v4f*>(p + (int64_t)heads * kHead);
      }
    }
  };
  auto commit = [&]() {
#pragma unroll
    for (int i = 0; i < kPasses; ++i) {
      const int row = lrow + i * step;
      if (row < kBlock) {
        *reinterpret_cast<v4f*>(&keys[row * kKeyPitch + lcol]) = kreg[i];
        *reinterpret_cast<v4f*>(&vals[row * kHead + lcol]) = vreg[i];
      }
    }
  };

  v4f o[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) o[t] = (v4f){0.f, 0.f, 0.f, 0.f};
  float m = -__builtin_inff(), l = 0.f;
  fetch(0);
  for (int key0 = 0; key0 < S; key0 += kBlock) {
    __syncthreads();                       // the block before has been read
    commit();
    __syncthreads();
    if (key0 + kBlock < S) fetch(key0 + kBlock);
    // scores of 64 keys, 16 per lane (already in units of log2)
    v4f s[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      s[kt] = (v4f){0.f, 0.f, 0.f, 0.f};
      if (key0 + kt * 16 >= S) continue;                    // (uniform: tiles past the sequence)
      const v4f* kp = reinterpret_cast<const v4f*>(&keys[(kt * 16 + r) * kKeyPitch + 16 * g]);
      v4f k[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) k[i] = kp[i];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) s[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][c], q[i][c], s[kt], 0, 0, 0);
    }
    float top = m;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (key0 + kt * 16 + 4 * g + v >= S) s[kt][v] = -__builtin_inff();
        top = fmaxf(top, s[kt][v]);
      }
    top = fmaxf(top, __shfl_xor(top, 16, 64));
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    // (scores of -inf alone so far: their probabilities are zero, where -inf - -inf would be a NaN for
    // the keys to come; nothing but -inf in the whole row divides zero by zero at the end)
    const float ref = top == -__builtin_inff() ? 0.f : top;
    const float keep = __builtin_amdgcn_exp2f(m - ref);     // (m = -inf at first: 0)
    m = top;
    float sum = 0.f;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[kt][v] = __builtin_amdgcn_exp2f(s[kt][v] - ref);
        sum += s[kt][v];
      }
    l = l * keep + sum;
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] *= keep;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      if (key0 + kt * 16 >= S) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const v4f vv = *reinterpret_cast<const v4f*>(&vals[(kt * 16 + 4 * g + v) * kHead + 4 * r]);
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[t], s[kt][v], o[t], 0, 0, 0);
      }
    }
  }
  // the four lanes of a query have each summed their own keys
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (q0 + r >= S) return;
  const float inv = 1.0f / l;
  // channel 16 g + 4 v + t is element v of tile t
  v4f y[4];
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int t = 0; t < 4; ++t) y[v][t] = o[t][v] * inv;
  store_context<QUANT>(y, ((int64_t)b * S + q0 + r) * heads * kHead + h * kHead + 16 * g, out, out_q, q_scale);
}

__device__ __forceinline__ float upper_half(float x) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & 0xffff0000u);
}
// the bf16 of two floats, cut off
__device__ __forceinline__ uint32_t upper_halves(float x, float y) {
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, y), __builtin_bit_cast(uint32_t, x), 0x07060302u);
}

// The same on the int8 result of the merged projection and its scale, for a layer whose projection is
// quantized: q, k and v are codes times one scale s, and nothing of them is widened to f32.
//  * S^T = K Q^T in whole numbers, one v_mfma_i32_16x16x64_i8 for 16 keys x 16 queries x 64 channels (in
//    f32 sixteen v_mfma_f32_16x16x4 of twice its time); lanes hold what they hold in the f32 kernel.  The
//    maxima are whole numbers too, and so is the difference in exp2((acc - max) f), f = s^2 log2(e) /
//    sqrt(64): at most 2^21, exact in f32.  The best key's probability is 1 whatever the scale.  (Of
//    max f, rounded, taken off acc f the best key keeps that rounding: several powers of two from scales
//    of 15 on, beyond the largest half.)
//  * O^T = V^T P^T on v_mfma_f32_16x16x32_bf16: a code is a bf16 as it is, and a probability the sum of
//    three, its 24 bits eight by eight, cut off and not rounded, so that every product is that of the f32
//    probability.  (Times 2^64: the last part of the smallest that the exponential gives is a normal number
//    then.  The sum of two halves has 22 to 24 of the bits and none below 2^-38 of the largest -- values
//    behind a key that has all the weight and is zero itself came out 1e-1 off at 2^-31 -- and is 0.3 us less
//    at 8 x 128 tokens, 2.5 at 8 x 384.)  24 instead of 128 matrix instructions for 64 keys, of half the time
//    each, and sums round a quarter as often: the rms error against 64 bits, over 24 scales from 0.003 to 0.3
//    at each of 8 to 384 tokens (300 where the codes are of three or five levels and one scale's few distinct
//    probabilities round one way), is 0.14 to 0.99 of the f32 kernel's on the dequantized projection, the smaller
//    the wider the scores spread; of the int8 results of eight encoder layers' attention 52 in 14.4 million
//    differ from those of 64 bits, with the f32 kernel 73.
//  * Values are widened and transposed once, on their way into LDS: a thread takes 4 channels of 4 keys.
//    A row of 64 keys is a channel, keys 32 j + 16 i + 4 g + v at 32 j + 8 g + 4 i + v, so that the eight
//    a lane multiplies are one 16-byte read; channel 4 r + t is row 16 t + r, 144 bytes apart, which spreads
//    the 16 channels of a read over all banks.  Keys lie in 64-byte rows, 16-byte chunk c of row r in slot
//    c ^ (r / 4 % 4), likewise.
//  * Two stages of 64 keys, one barrier a block.  Always four waves: those past a short sequence's queries
//    multiply copies, but load and widen their part of the keys and values (1 x 8 tokens 3.3 us, the f32
//    kernel on one wave 5.4).
// What is left is the vector work of the softmax, fourteen instructions per score, and at encoder sizes the
// launch and the trips to memory.  us, one after the other in a graph, this kernel / the f32 one: 12 heads of
// 8 x 128 tokens 4.8 / 9.7, 4 x 336 11.0 / 31.8, 8 x 384 15.4 / 49.0; the projection in front of it 7.6 / 10.4 at
// 8 x 128 (2.4 MB of int8 results in place of 9.4 MB of f32).
template <bool QUANT>
__global__ void __launch_bounds__(256, 2)
attention_i8_kernel(const int8_t* __restrict__ qkv, const float* __restrict__ qkv_scale, int S, uint32_t all_heads,
                    int heads, float* __restrict__ out, int8_t* __restrict__ out_q,
                    const float* __restrict__ q_scale) {
  constexpr int kValPitch = 144, kStage = kBlock * kHead + kHead * kValPitch;     // bytes
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * kStage];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const uint32_t bh = blockIdx.x % all_heads, tile = blockIdx.x / all_heads;
  const int b = (int)(bh / heads), h = (int)(bh % heads);
  const uint32_t row3 = 3u * (uint32_t)heads * kHead;        // bytes between two tokens
  const int8_t* base = qkv + (int64_t)b * S * row3 + (int64_t)h * kHead;
  auto token = [&](int row) { return (uint64_t)(uint32_t)min(row, S - 1) * row3; };
  const int q0 = ((int)tile * 4 + wave) * 16;

  const v4i q = *reinterpret_cast<const v4i*>(base + token(q0 + r) + 16 * g);
  const float s = qkv_scale[0];
  const float f = s * s * (1.4426950408889634f / 8.0f);      // log2(e) / sqrt(64)

  // (copies of the last token past the sequence: their probabilities are set to zero)
  const int krow = threadIdx.x >> 2, kchunk = threadIdx.x & 3, vc = threadIdx.x & 15, vk = threadIdx.x >> 4;
  const int8_t* kbase = base + (int64_t)heads * kHead + 16 * kchunk;
  const int8_t* vbase = base + 2 * (int64_t)heads * kHead + 4 * vc;
  uint8_t* kdst = lds + krow * kHead + 16 * (kchunk ^ ((krow >> 2) & 3));
  uint8_t* vdst = lds + kBlock * kHead + vc * kValPitch + 2 * (32 * (vk >> 3) + 8 * (vk & 3) + 4 * ((vk >> 2) & 1));
  v4i kreg;
  uint32_t vreg[4];
  auto fetch = [&](int key0) {
    kreg = *reinterpret_cast<const v4i*>(kbase + token(key0 + krow));
#pragma unroll
    for (int i = 0; i < 4; ++i)
      vreg[i] = *reinterpret_cast<const uint32_t*>(vbase + token(key0 + 4 * vk + i));
  };
  auto commit = [&](int stage) {
    *reinterpret_cast<v4i*>(kdst + stage * kStage) = kreg;
#pragma unroll
    for (int t = 0; t < 4; ++t) {                            // channel 4 vc + t of four keys
      uint32_t w[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        w[i] = upper_halves((float)(int8_t)(vreg[2 * i] >> (8 * t)), (float)(int8_t)(vreg[2 * i + 1] >> (8 * t)));
      *reinterpret_cast<uint2*>(vdst + stage * kStage + 16 * t * kValPitch) = make_uint2(w[0], w[1]);
    }
  };

  v4f o[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) o[t] = (v4f){0.f, 0.f, 0.f, 0.f};
  int m = -kHead * 128 * 128;                                // (no sum of 64 products is below it)
  float l = 0.f;
  fetch(0);
  commit(0);
  if (kBlock < S) fetch(kBlock);
  __syncthreads();
  int stage = 0;
  for (int key0 = 0; key0 < S; key0 += kBlock, stage ^= 1) {
    const uint8_t* kp = lds + stage * kStage + r * kHead + 16 * (g ^ ((r >> 2) & 3));
    const uint8_t* vp = lds + stage * kStage + kBlock * kHead + r * kValPitch + 16 * g;
    v4i a[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
      a[kt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i*>(kp + kt * 16 * kHead), q,
                                                    (v4i){0, 0, 0, 0}, 0, 0, 0);
    const bool ragged = key0 + kBlock > S;
    int top = m;
    if (!ragged) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int v = 0; v < 4; ++v) top = max(top, a[kt][v]);
    } else {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int v = 0; v < 4; ++v) top = key0 + kt * 16 + 4 * g + v < S ? max(top, a[kt][v]) : top;
    }
    {  // over the four lanes of a query
      auto x = __builtin_amdgcn_permlane16_swap(top, top, false, false);
      top = max((int)x[0], (int)x[1]);
      x = __builtin_amdgcn_permlane32_swap(top, top, false, false);
      top = max((int)x[0], (int)x[1]);
    }
    const float keep = __builtin_amdgcn_exp2f((float)(m - top) * f);
    m = top;
    float p[4][4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        p[kt][v] = __builtin_amdgcn_exp2f((float)(a[kt][v] - top) * f) * 0x1p64f;
    if (ragged) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int v = 0; v < 4; ++v) p[kt][v] = key0 + kt * 16 + 4 * g + v < S ? p[kt][v] : 0.f;
    }
    float sum = 0.f;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) sum += (p[kt][0] + p[kt][1]) + (p[kt][2] + p[kt][3]);
    l = l * keep + sum;
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] *= keep;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (key0 + 32 * j >= S) continue;                      // (uniform: keys past the sequence)
      v4i part[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x = p[2 * j + (e >> 1)][2 * (e & 1)], y = p[2 * j + (e >> 1)][2 * (e & 1) + 1];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          part[c][e] = (int)upper_halves(x, y);
          x -= upper_half(x);                  // (exact)
          y -= upper_half(y);
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const b8 vv = *reinterpret_cast<const b8*>(vp + 16 * t * kValPitch + 64 * j);
#pragma unroll
        for (int c = 0; c < 3; ++c)
          o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, __builtin_bit_cast(b8, part[c]), o[t], 0, 0, 0);
      }
    }
    if (key0 + kBlock < S) {
      commit(stage ^ 1);                     // (last read before the barrier of the block before)
      if (key0 + 2 * kBlock < S) fetch(key0 + 2 * kBlock);
      __syncthreads();
    }
  }
  // the four lanes of a query have each summed their own keys
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (q0 + r >= S) return;
  const float inv = s / (l * 0x1p-64f);
  // channel 16 g + 4 v + t is element v of tile t
  v4f y[4];
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int t = 0; t < 4; ++t) y[v][t] = (o[t][v] * 0x1p-64f) * inv;
  store_context<QUANT>(y, ((int64_t)b * S + q0 + r) * heads * kHead + h * kHead + 16 * g, out, out_q, q_scale);
}

// ------------------------------------------------------------------ layer normalisation
// A wave per row, up to 2048 columns in its registers: mean, then the variance of the differences,
// then (x - mean) * rstd * gamma + beta, written as f32, quantized, or both -- the row is read once
// and the quantize that follows costs its one byte per element.  Bound by the launch at encoder
// sizes (1024 x 768: 3 MB read).
template <int N4, bool QUANT>
__global__ void __launch_bounds__(256)
layernorm_f32_kernel(const float* __restrict__ x, int64_t rows, int cols, const float* __restrict__ gamma,
                     const float* __restrict__ beta, float eps, float* __restrict__ out,
                     int8_t* __restrict__ out_q, const float* __restrict__ q_scale) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const v4f* p = reinterpret_cast<const v4f*>(x + row * cols);
  const int n4 = cols >> 2;
  v4f v[N4];
#pragma unroll
  for (int i = 0; i < N4; ++i) v[i] = lane + 64 * i < n4 ? p[lane + 64 * i] : (v4f){0.f, 0.f, 0.f, 0.f};
  v4f ga[N4], be[N4];
#pragma unroll
  for (int i = 0; i < N4; ++i) {
    const int c = lane + 64 * i < n4 ? lane + 64 * i : 0;
    ga[i] = reinterpret_cast<const v4f*>(gamma)[c];
    be[i] = reinterpret_cast<const v4f*>(beta)[c];
  }
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < N4; ++i) sum += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  const float mean = sum / (float)cols;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < N4; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = lane + 64 * i < n4 ? v[i][e] - mean : 0.f;
      v[i][e] = d;
      sq += d * d;
    }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off, 64);
  const float rstd = 1.0f / __builtin_sqrtf(sq / (float)cols + eps);
  float sc = 1.f, rcp = 1.f;
  bool fast = true;
  if (QUANT) {
    sc = q_scale[0];
    rcp = 1.0f / sc;
    fast = elementwise::divisor_in_fast_range(sc);
  }
#pragma unroll
  for (int i = 0; i < N4; ++i) {
    if (lane + 64 * i >= n4) continue;
    const v4f y = v[i] * rstd * ga[i] + be[i];
    if (out) reinterpret_cast<v4f*>(out + row * cols)[lane + 64 * i] = y;
    if (QUANT) reinterpret_cast<uint32_t*>(out_q + row * cols)[lane + 64 * i] = quantize4(y, sc, rcp, fast);
  }
}

template <int N4>
void launch_layernorm(const float* x, int64_t rows, int cols, const float* gamma, const float* beta, float eps,
                      float* out, int8_t* out_q, const float* q_scale, hipStream_t st) {
  const dim3 grid((unsigned)ceil_div(rows, 4)), block(256);
  if (out_q)
    hipLaunchKernelGGL((layernorm_f32_kernel<N4, true>), grid, block, 0, st, x, rows, cols, gamma, beta, eps, out,
                       out_q, q_scale);
  else
    hipLaunchKernelGGL((layernorm_f32_kernel<N4, false>), grid, block, 0, st, x, rows, cols, gamma, beta, eps,
                       out, out_q, q_scale);
}

}  // namespace
}  // namespace dq8

using namespace dq8;

extern "C" int dq8_attention_f32(const float* qkv, int64_t batch, int64_t seq, int64_t heads,
                                 int64_t head_dim, float* out, int8_t* out_q, const float* q_scale,
                                 void* stream) {
  clear_error();
  DQ8_REQUIRE(batch >= 0 && seq >= 0 && heads >= 0, "dq8_attention_f32: negative size");
  DQ8_REQUIRE(head_dim == kHead, "dq8_attention_f32: heads of 64 channels only");
  if (batch == 0 || seq == 0 || heads == 0) return 0;
  DQ8_REQUIRE(qkv && (out || out_q), "dq8_attention_f32: null pointer");
  DQ8_REQUIRE(!(out && out_q) && (!out_q || q_scale), "dq8_attention_f32: an f32 result, or an int8 one and its scale");
  DQ8_REQUIRE(aligned(qkv, 16) && aligned(out, 16) && aligned(out_q, 16), "dq8_attention_f32: 16-byte aligned tensors");
  // waves of 16 queries: four to a workgroup, fewer for a short sequence
  const int waves = (int)(seq >= 49 ? 4 : ceil_div(seq, 16));
  const int64_t tiles = ceil_div(seq, 16 * waves);
  DQ8_REQUIRE(seq < (1 << 24) && batch < (1 << 24) && heads < (1 << 24) && batch * heads < (1LL << 31) / tiles,
              "dq8_attention_f32: too large");
  const dim3 grid((unsigned)(batch * heads * tiles)), block(64 * waves);
  const float scale_log2 = 1.4426950408889634f / 8.0f;      // log2(e) / sqrt(64)
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, block, 0, (hipStream_t)stream, qkv, (int)seq, (uint32_t)(batch * heads), (int)heads, scale_log2, out, out_q,
                       q_scale);
  };
  switch (waves) {
    case 1: launch(out_q ? attention_f32_kernel<1, true> : attention_f32_kernel<1, false>); break;
    case 2: launch(out_q ? attention_f32_kernel<2, true> : attention_f32_kernel<2, false>); break;
    case 3: launch(out_q ? attention_f32_kernel<3, true> : attention_f32_kernel<3, false>); break;
    default: launch(out_q ? attention_f32_kernel<4, true> : attention_f32_kernel<4, false>); break;
  }
  return check_hip(hipGetLastError(), "dq8_attention_f32 launch");
}

extern "C" int dq8_attention_i8(const int8_t* qkv, const float* qkv_scale, int64_t batch, int64_t seq,
                                int64_t heads, int64_t head_dim, float* out, int8_t* out_q,
                                const float* q_scale, void* stream) {
  clear_error();
  DQ8_REQUIRE(batch >= 0 && seq >= 0 && heads >= 0, "dq8_attention_i8: negative size");
  DQ8_REQUIRE(head_dim == kHead, "dq8_attention_i8: heads of 64 channels only");
  if (batch == 0 || seq == 0 || heads == 0) return 0;
  DQ8_REQUIRE(qkv && qkv_scale && (out || out_q), "dq8_attention_i8: null pointer");
  DQ8_REQUIRE(!(out && out_q) && (!out_q || q_scale), "dq8_attention_i8: an f32 result, or an int8 one and its scale");
  DQ8_REQUIRE(aligned(qkv, 16) && aligned(out, 16) && aligned(out_q, 16), "dq8_attention_i8: 16-byte aligned tensors");
  const int64_t tiles = ceil_div(seq, 64);
  DQ8_REQUIRE(seq < (1 << 24) && batch < (1 << 24) && heads < (1 << 24) && batch * heads < (1LL << 31) / tiles,
              "dq8_attention_i8: too large");
  const dim3 grid((unsigned)(batch * heads * tiles)), block(256);
  if (out_q)
    hipLaunchKernelGGL(attention_i8_kernel<true>, grid, block, 0, (hipStream_t)stream, qkv, qkv_scale, (int)seq,
                       (uint32_t)(batch * heads), (int)heads, out, out_q, q_scale);
  else
    hipLaunchKernelGGL(attention_i8_kernel<false>, grid, block, 0, (hipStream_t)stream, qkv, qkv_scale, (int)seq,
                       (uint32_t)(batch * heads), (int)heads, out, out_q, q_scale);
  return check_hip(hipGetLastError(), "dq8_attention_i8 launch");
}

extern "C" int dq8_layernorm_f32(const float* x, int64_t rows, int64_t cols, const float* gamma,
                                 const float* beta, float eps, float* out, int8_t* out_q,
                                 const float* q_scale, void* stream) {
  clear_error();
  DQ8_REQUIRE(rows >= 0 && cols >= 0, "dq8_layernorm_f32: negative size");
  if (rows == 0 || cols == 0) return 0;
  DQ8_REQUIRE(cols % 4 == 0 && cols <= 2048, "dq8_layernorm_f32: up to 2048 columns, a multiple of 4");
  DQ8_REQUIRE(x && gamma && beta && (out || out_q) && (!out_q || q_scale), "dq8_layernorm_f32: null pointer");
  DQ8_REQUIRE(aligned(x, 16) && aligned(gamma, 16) && aligned(beta, 16) && aligned(out, 16) && aligned(out_q, 4),
              "dq8_layernorm_f32: 16-byte aligned tensors");
  DQ8_REQUIRE(rows < (1LL << 32), "dq8_layernorm_f32: too many rows");
  hipStream_t st = (hipStream_t)stream;
  const int n = (int)ceil_div(cols, 256);
  if (n <= 1) launch_layernorm<1>(x, rows, (int)cols, gamma, beta, eps, out, out_q, q_scale, st);
  else if (n <= 3) launch_layernorm<3>(x, rows, (int)cols, gamma, beta, eps, out, out_q, q_scale, st);
  else if (n == 4) launch_layernorm<4>(x, rows, (int)cols, gamma, beta, eps, out, out_q, q_scale, st);
  else launch_layernorm<8>(x, rows, (int)cols, gamma, beta, eps, out, out_q, q_scale, st);
  return check_hip(hipGetLastError(), "dq8_layernorm_f32 launch");
}
