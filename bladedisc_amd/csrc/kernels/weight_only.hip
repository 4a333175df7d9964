// Weight-only quantized GEMM for gfx950: floating-point activations (f16 or f32) times 8-bit
// weights with a per-output-channel scale and zero point,
//
//   out[m, n] = (sum_k x[m, k] * (w[n, k] - zp[n])) * scale[n] + bias[n]
//
// which is matmul(x, dequantize(w)^T) + bias with the scale taken out of the sum.  This is the
// runtime side of the reference's `ral_pdll_weight_only_qgemm` custom call
// (pytorch_blade/tests/disc/pdl/pdll_files/gpu/weight_only_qgemm.pdll:2-104; operands input,
// weight ui8 [K, N], [bias,] weight_scale, weight_zero_point), for which the reference tree
// holds no implementation.
//
// The weights stay 8-bit in memory and are widened on their way into the matrix cores
// (v_mfma_f32_32x32x16_f16, f32 accumulation): a byte b becomes the half 0x6400 | b = 1024 + b
// with one v_perm_b32 per two weights, and one packed subtraction of 1024 + zp[n] leaves
// b - zp[n] exactly (|b - zp| <= 2048 is an integer a half holds).  Products of a half
// activation (11 significant bits) and such a weight (9 bits) are exact in f32, so the only
// rounding is the f32 accumulation.  f32 activations are split into two halves
// x = hi + lo (hi = half(x), lo = half(x - hi)) and both are multiplied: about 22 significant
// bits of x take part while lo is a normal half (|x| >= 1/8); below, lo is subnormal and the
// error per activation is an absolute 2^-25.
//
// In the register kernels both operands go from global memory straight into registers in MFMA
// layout: the order of the k values inside a fragment is free as long as both operands agree,
// so lane (row, g) takes the 16 consecutive k values k0 + 16 g .. of its row -- 16 weight bytes
// (one dwordx4), 16 activations -- and feeds two MFMAs with them.
//  * wo_dma_kernel: tiles loaded straight into LDS, everything above 32 rows (16 for f32 against deep or
//    wide weights, f32_rows_on_tiles): 32 x 64 to 128 x 256 tiles, with several workgroups per tile, each
//    over a part of k, and wo_splitk_reduce_kernel behind them, where that is estimated cheaper (1.1-1.2
//    PFLOP/s for f16 activations at 4096^2 .. 8192^2 weights, where the ROCm library's plain f16 GEMM
//    reaches 1.16-1.49);
//  * wo_ragged_kernel: the same for f16 rows that begin at any byte, through registers;
//  * wo_tile_kernel: 2 x 2 waves, wave tile (32 FM) x (32 FN), operands straight into registers:
//    operands too large for the LDS kernel's 31-bit offsets;
//  * wo_rows_kernel: 2 .. 32 rows, 16 .. 64 output channels per workgroup, both operands loaded in
//    row segments and turned into fragments through wave-private LDS;
//  * wo_gemv_kernel: one or two rows, a wave per output channel streaming its weight row on the
//    vector ALUs;
//  * wo_skinny_kernel: M <= 128 rows against 32 output channels per workgroup, the k range dealt
//    over the waves and the partial sums added through LDS: operands too large for the LDS
//    kernels' 31-bit offsets;
//  * wo_exact_f32_kernel: f32 activations on rows off 16 bytes (f16 ones: wo_ragged_kernel, and
//    wo_rows_kernel's RAGGED form up to 32 rows);
//  * wo_generic_kernel: one output per thread, fewer than 16 of k or weights left as [K, N].
#include <algorithm>
#include <type_traits>
#include <utility>

#include "dq8_common.h"
#include "disc_q8.h"
#include "lds_direct.h"

#pragma clang fp contract(off)

namespace dq8 {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

struct WoParams {
  const void* x;        // [M, K] activations, row stride ldx elements
  const uint8_t* w;     // weights; element (n, k) at w[n * w_sn + k * w_sk]
  const void* scale;    // [N], activation dtype
  const int32_t* zp;    // [N] or null (zero)
  const void* bias;     // [N] or null, activation dtype
  void* out;            // [M, N], row stride ldo elements
  int64_t ldx, ldo, w_sn, w_sk;
  int M, N, K;
  unsigned flip;        // 0x80808080 for signed weights (b ^ 0x80 = b + 128 as unsigned)
  // split k (wo_dma_kernel, wo_ragged_kernel): workgroup (tile, y) multiplies k in [y k_split, (y + 1) k_split)
  // and, when `partial` is set, leaves its f32 sums in partial[y][M][N] for the reduction kernel
  float* partial;
  int k_split;          // a multiple of 64; K when the k range is not split
  bool ragged;          // rows that are not multiples of 16 bytes, 16-byte aligned
  bool words;           // (f16) ... but begin on four bytes, K % 4 == 0
};

// RAGGED kernels: rows of any length from 16 on and any alignment.  A row's 16-element chunk that
// is not whole is read as the row's last 16 elements, of both operands, and the activations that a
// chunk before it holds already are made zero (the weights that meet them are finite).
typedef unsigned u4_any __attribute__((ext_vector_type(4), aligned(1)));
__device__ __forceinline__ u4 load_any(const uint8_t* base, unsigned off) {
  return *reinterpret_cast<const u4_any*>(base + off);
}
// the first z of eight halves made zero
__device__ __forceinline__ u4 zero_first(u4 q, int z) {
#pragma unroll
  for (int d = 0; d < 4; ++d) q[d] = z >= 2 * d + 2 ? 0u : z == 2 * d + 1 ? q[d] & 0xffff0000u : q[d];
  return q;
}

// body(Int<0>()), ..., body(Int<N - 1>())
template <int V>
using Int = std::integral_constant<int, V>;
template <typename Body, int... I>
__device__ __forceinline__ void static_for_seq(Body&& body, std::integer_sequence<int, I...>) {
  (body(Int<I>()), ...);
}
template <int N, typename Body>
__device__ __forceinline__ void static_for_n(Body&& body) {
  static_for_seq(body, std::make_integer_sequence<int, N>());
}

template <typename T>
__device__ __forceinline__ float to_f32(T v) {
  return (float)v;
}

// 16 weight bytes -> the halves of two MFMA k-steps, minus c = 1024 + zp (+128 if signed)
__device__ __forceinline__ void widen16(u4 q, unsigned flip, h2 c, h8& s0, h8& s1) {
  auto pair = [&](unsigned d, unsigned sel) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, d ^ flip, sel)) - c;
  };
  const h2 a0 = pair(q.x, 0x05010400u), a1 = pair(q.x, 0x07030602u);
  const h2 a2 = pair(q.y, 0x05010400u), a3 = pair(q.y, 0x07030602u);
  const h2 b0 = pair(q.z, 0x05010400u), b1 = pair(q.z, 0x07030602u);
  const h2 b2 = pair(q.w, 0x05010400u), b3 = pair(q.w, 0x07030602u);
  s0 = (h8){a0.x, a0.y, a1.x, a1.y, a2.x, a2.y, a3.x, a3.y};
  s1 = (h8){b0.x, b0.y, b1.x, b1.y, b2.x, b2.y, b3.x, b3.y};
}

// eight of them: one k-step
__device__ __forceinline__ h8 widen8(unsigned d0, unsigned d1, unsigned flip, h2 c) {
  auto pair = [&](unsigned d, unsigned sel) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, d ^ flip, sel)) - c;
  };
  const h2 a0 = pair(d0, 0x05010400u), a1 = pair(d0, 0x07030602u);
  const h2 a2 = pair(d1, 0x05010400u), a3 = pair(d1, 0x07030602u);
  return (h8){a0.x, a0.y, a1.x, a1.y, a2.x, a2.y, a3.x, a3.y};
}

// x = hi + lo of two activations, hi = half(x), lo = half(x - hi).  x - hi is exact, as a difference
// and as the fused multiply-add that reads the half where it is: four instructions for two values
// in place of eight.
__device__ __forceinline__ void split2(float x, float y, h2& hi, h2& lo) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  hi = __builtin_convertvector((f2){x, y}, h2);
#if defined(__HIP_DEVICE_COMPILE__)
  f2 d;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d.x) : "v"(hi), "v"(x));
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d.y) : "v"(hi), "v"(y));
#else
  const f2 d = {x - (float)hi.x, y - (float)hi.y};
#endif
  lo = __builtin_convertvector(d, h2);
}

// The 16 activations of a lane for one 32-deep k chunk: two k-steps, and for f32 activations a
// second pair holding what the first rounded away.
template <typename XT>
struct XFrag;

template <>
struct XFrag<_Float16> {
  u4 r0, r1;
  static constexpr int kParts = 1;
  __device__ __forceinline__ void load(const _Float16* p, bool valid) {
    const u4 z = {0, 0, 0, 0};
    r0 = valid ? *reinterpret_cast<const u4*>(p) : z;
    r1 = valid ? *reinterpret_cast<const u4*>(p + 8) : z;
  }
  __device__ __forceinline__ h8 step(int part, int s) const {
    (void)part;
    return __builtin_bit_cast(h8, s == 0 ? r0 : r1);
  }
};

template <>
struct XFrag<float> {
  f4 r[4];
  static constexpr int kParts = 2;
  __device__ __forceinline__ void load(const float* p, bool valid) {
    const f4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = valid ? *reinterpret_cast<const f4*>(p + 4 * i) : z;
  }
  __device__ __forceinline__ h8 step(int part, int s) const {
    h8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = r[2 * s + e / 4][e % 4];
      const _Float16 hi = (_Float16)v;
      o[e] = part == 0 ? hi : (_Float16)(v - (float)hi);
    }
    return o;
  }
};

template <typename XT>
__device__ __forceinline__ void store_frag(const WoParams& p, const f16v& acc, int m_base, int n,
                                           int lane) {
  if (n >= p.N) return;
  const XT* scale = static_cast<const XT*>(p.scale);
  const XT* bias = static_cast<const XT*>(p.bias);
  const float s = to_f32(scale[n]);
  const float b = bias ? to_f32(bias[n]) : 0.0f;
  XT* out = static_cast<XT*>(p.out);
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int m = m_base + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
    if (m < p.M) out[(int64_t)m * p.ldo + n] = (XT)(acc[v] * s + b);
  }
}

// The raw sums of one k range, for wo_splitk_reduce_kernel.
__device__ __forceinline__ void store_partial(const WoParams& p, const f16v& acc, int split,
                                              int m_base, int n, int lane) {
  if (n >= p.N) return;
  float* dst = p.partial + (int64_t)split * p.M * p.N;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int m = m_base + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
    if (m < p.M) dst[(int64_t)m * p.N + n] = acc[v];
  }
}

__device__ __forceinline__ h2 centre(const WoParams& p, int n) {
  const int zp = p.zp ? p.zp[n] : 0;
  const _Float16 c = (_Float16)(float)(1024 + zp + (p.flip ? 128 : 0));
  return (h2){c, c};
}

// ---------------------------------------------------------------- tiled kernel, M > 32
template <typename XT, int FM, int FN>
__global__ void __launch_bounds__(256) wo_tile_kernel(const WoParams p) {
  constexpr int BM = 2 * FM * 32, BN = 2 * FN * 32;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_n = (p.N + BN - 1) / BN;
  const int m0 = (blockIdx.x / tiles_n) * BM + wm * FM * 32;
  const int n0 = (blockIdx.x % tiles_n) * BN + wn * FN * 32;
  const int r = lane & 31, g = lane >> 5;

  const XT* xrow[FM];
  const uint8_t* wrow[FN];
  h2 c[FN];
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = min(m0 + i * 32 + r, p.M - 1);          // rows past M re-read the last one
    xrow[i] = static_cast<const XT*>(p.x) + (int64_t)m * p.ldx + 16 * g;
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = min(n0 + j * 32 + r, p.N - 1);
    wrow[j] = p.w + (int64_t)n * p.w_sn + 16 * g;
    c[j] = centre(p, n);
  }
  f16v acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // D chunks of 32 in flight per wave (registers permitting: f32 activations take twice the
  // registers of f16 ones)
  constexpr int D = sizeof(XT) == 2 ? 4 : 2;
  XFrag<XT> xr[D][FM];
  u4 wr[D][FN];
  const u4 zero = {0, 0, 0, 0};
  auto load = [&](XFrag<XT>* xf, u4* wf, int k0) {
    const bool valid = k0 + 16 * g < p.K;                // K % 16 == 0: whole 16-chunks
    const int k = valid ? k0 : 0;
#pragma unroll
    for (int i = 0; i < FM; ++i) xf[i].load(xrow[i] + k, valid);
#pragma unroll
    for (int j = 0; j < FN; ++j) wf[j] = valid ? *reinterpret_cast<const u4*>(wrow[j] + k) : zero;
  };
  auto compute = [&](const XFrag<XT>* xf, const u4* wf) {
    h8 w0[FN], w1[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) widen16(wf[j], p.flip, c[j], w0[j], w1[j]);
#pragma unroll
    for (int part = 0; part < XFrag<XT>::kParts; ++part)
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const h8 a0 = xf[i].step(part, 0), a1 = xf[i].step(part, 1);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, w0[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, w1[j], acc[i][j], 0, 0, 0);
        }
      }
  };
  // a ring of D chunks: each is multiplied and at once refilled with the chunk D further on,
  // so D - 1 loads stay in flight under every multiplication (one chunk ahead measured 16 % of
  // the matrix rate: a wave waited out the whole load latency per chunk)
#pragma unroll
  for (int d = 0; d < D; ++d) load(xr[d], wr[d], d * 32);
  for (int k0 = 0; k0 < p.K; k0 += D * 32) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      compute(xr[d], wr[d]);
      load(xr[d], wr[d], k0 + (D + d) * 32);             // (past K: zeros)
    }
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
      store_frag<XT>(p, acc[i][j], m0 + i * 32, n0 + j * 32 + r, lane);
}

// ---------------------------------------------------------------- f16 rows of any length: tiles through registers and LDS
// (32 WM) x (64 FN) tile, WM x 2 waves of 32 x (32 FN), k tiles of 64 in two LDS stages.  Eight lanes
// cover one 128-byte row segment of the activations and four one 64-byte segment of the weights, by
// loads of any alignment; the tile is shared through LDS (16-byte chunks XOR-swizzled by the row so
// that the fragment reads spread over the banks) and the fragments are read back as ds_read_b128.
// The weights are widened to halves once, on their way into LDS (128-byte rows like the
// activations'), not by every wave that reads them.  Only the k tile with the end of the rows is
// handled differently (M = 512, 2047 -> 3001, one output per thread before: 11.9 ms).
//
// Four register sets hold the k tiles t + 1 .. t + 4 on their way from memory while tile t is
// multiplied.  The loads have no branch around them and the main loop is four k tiles of
// straight-line code, so that the wait in front of a tile's hand-over to LDS counts the loads
// issued after it instead of draining them all: with conditional loads in a loop of guarded steps
// every k tile waited out a whole trip to memory (0.8 us per k tile on a quiet chip, 1.5-2 us on a
// busy one).
template <int WM, int FN>
__global__ void __launch_bounds__(WM * 128, 2) wo_ragged_kernel(const WoParams p) {
  constexpr int BM = WM * 32, BN = 2 * FN * 32, BK = 64, SETS = 4;
  constexpr int NT = WM * 128;                           // WM x 2 waves
  constexpr int XP = (BM * 8) / NT;                      // activation chunks per thread
  constexpr int WP = (BN * 4) / NT;                      // weight chunks per thread
  constexpr int XS = BM * 128;                           // activation bytes of a stage
  static_assert(SETS % 2 == 0 && SETS * (XP + WP) <= 63, "two LDS stages; vmcnt has 6 bits");
  // two stages of (activation tile, widened weight tile), 128 bytes per row
  extern __shared__ __attribute__((aligned(1024))) uint8_t wo_lds[];
  uint8_t* const xs[2] = {wo_lds, wo_lds + XS};
  uint8_t* const ws[2] = {wo_lds + 2 * XS, wo_lds + 2 * XS + BN * 128};
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_n = (p.N + BN - 1) / BN;
  // Workgroups go to the 8 XCDs round-robin, and each XCD has its own L2.  Where the tile grid
  // divides, XCD x takes one compact patch of it (the grid cut 4 x 2: an activation row is
  // twice the bytes of a weight row), so that its L2 fetches the patch's operand rows instead
  // of every activation row.
  int tile = blockIdx.x;
  {
    const int tiles_m = gridDim.x / tiles_n;
    // (launches of at least a round; the rows of a split launch are not dealt this way)
    if (gridDim.y == 1 && gridDim.x >= 128 && tiles_m % 4 == 0 && tiles_n % 2 == 0) {
      const int xcd = tile & 7, idx = tile >> 3;
      const int pm = tiles_m / 4, pn = tiles_n / 2;        // the patch
      tile = ((xcd >> 1) * pm + idx / pn) * tiles_n + (xcd & 1) * pn + idx % pn;
    }
  }
  const int m0 = (tile / tiles_n) * BM, n0 = (tile % tiles_n) * BN;
  const int r = lane & 31, g = lane >> 5;
  const int kbeg = blockIdx.y * p.k_split;               // this workgroup's k range
  const int klen = min(p.K, kbeg + p.k_split) - kbeg;
  const int mrows = min(BM, p.M - m0), nrows = min(BN, p.N - n0);

  // global -> LDS assignment (rows past the tile's last re-read that one; the host has checked that
  // the offsets fit 31 bits)
  const int xc = tid & 7, wc = tid & 3;                  // 16-byte chunk of the row's k tile
  int xo[XP], xl[XP];
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int row = tid / 8 + (NT / 8) * i;
    const int sx = (row ^ (row >> 3)) & 7;
    xo[i] = (int)((int64_t)min(row, mrows - 1) * p.ldx * 2);
    xl[i] = row * 128 + ((xc ^ sx) << 4);
  }
  int wo[WP], wl[WP], wl1[WP];
  h2 cpark[WP];
#pragma unroll
  for (int i = 0; i < WP; ++i) {
    const int row = (tid >> 2) + (NT / 4) * i;
    const int sw = (row ^ (row >> 3)) & 7;
    wo[i] = (int)((int64_t)min(row, nrows - 1) * p.w_sn);
    wl[i] = row * 128 + (((2 * wc) ^ sw) << 4);
    wl1[i] = row * 128 + (((2 * wc + 1) ^ sw) << 4);
    cpark[i] = centre(p, n0 + min(row, nrows - 1));
  }
  u4 xr[SETS][XP], wr[SETS][WP];
  const uint8_t* xbase = reinterpret_cast<const uint8_t*>(static_cast<const _Float16*>(p.x) + (int64_t)m0 * p.ldx);
  const uint8_t* wbase = p.w + (int64_t)n0 * p.w_sn;
  auto fetch = [&](u4* xq, u4* wq, int k0) {
    const unsigned kx = min(kbeg + k0 + 16 * (xc >> 1), p.K - 16) + 8 * (xc & 1);
    const unsigned kw = min(kbeg + k0 + 16 * wc, p.K - 16);
#pragma unroll
    for (int i = 0; i < XP; ++i) xq[i] = load_any(xbase, (unsigned)xo[i] + 2 * kx);
#pragma unroll
    for (int i = 0; i < WP; ++i) wq[i] = load_any(wbase, (unsigned)wo[i] + kw);
  };
  auto park = [&](u4* xq, const u4* wq, int stage, int k0) {
    if (k0 + BK > klen) {                                  // (uniform) the end of the rows
      const int c16 = kbeg + k0 + 16 * (xc >> 1);
      const int z = c16 - min(c16, p.K - 16) - 8 * (xc & 1);
#pragma unroll
      for (int i = 0; i < XP; ++i) xq[i] = zero_first(xq[i], z);
    }
#pragma unroll
    for (int i = 0; i < XP; ++i) *reinterpret_cast<u4*>(&xs[stage][xl[i]]) = xq[i];
#pragma unroll
    for (int i = 0; i < WP; ++i) {
      h8 lo, hi;
      widen16(wq[i], p.flip, cpark[i], lo, hi);
      *reinterpret_cast<h8*>(&ws[stage][wl[i]]) = lo;
      *reinterpret_cast<h8*>(&ws[stage][wl1[i]]) = hi;
    }
  };

  // fragment rows of this wave
  const int xrow = wm * 32 + r;
  int wrow[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) wrow[j] = (wn * FN + j) * 32 + r;
  f16v acc[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.0f;
  auto multiply = [&](int st) {
    const int sx = (xrow ^ (xrow >> 3)) & 7;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int c0 = 4 * s + 2 * g;
      const h8 a0 = *reinterpret_cast<const h8*>(&xs[st][xrow * 128 + ((c0 ^ sx) << 4)]);
      const h8 a1 = *reinterpret_cast<const h8*>(&xs[st][xrow * 128 + (((c0 + 1) ^ sx) << 4)]);
      h8 w0[FN], w1[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int row = wrow[j], sw = (row ^ (row >> 3)) & 7;
        w0[j] = *reinterpret_cast<const h8*>(&ws[st][row * 128 + ((c0 ^ sw) << 4)]);
        w1[j] = *reinterpret_cast<const h8*>(&ws[st][row * 128 + (((c0 + 1) ^ sw) << 4)]);
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, w0[j], acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, w1[j], acc[j], 0, 0, 0);
      }
    }
  };
  // k tile t: set u = t % SETS has been handed to LDS stage t % 2 and takes tile t + SETS;
  // tile t + 1 is handed over behind the multiplication
  // (the scheduling barriers keep a later step's arithmetic on loaded registers -- the first
  // instructions of widening -- from being moved up to where it would wait for their loads.  Between
  // a multiplication and the hand-over behind it there is none: the tile handed over left memory
  // SETS - 1 tiles ago, and its widening and writes fill the gaps between the MFMAs.)
  auto step = [&](int u, int t) {
    fetch(xr[u], wr[u], (t + SETS) * BK);
    multiply(u % 2);
    park(xr[(u + 1) % SETS], wr[(u + 1) % SETS], (u + 1) % 2, (t + 1) * BK);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
  };
  const int KT = (klen + BK - 1) / BK;
#pragma unroll
  for (int d = 0; d < SETS; ++d) fetch(xr[d], wr[d], d * BK);
  __builtin_amdgcn_sched_barrier(0);
  park(xr[0], wr[0], 0, 0);
  __syncthreads();
  __builtin_amdgcn_sched_barrier(0);
  int t = 0;
  for (; t + SETS <= KT; t += SETS) {
#pragma unroll
    for (int u = 0; u < SETS; ++u) step(u, t + u);
  }
#pragma unroll
  for (int u = 0; u < SETS - 1; ++u)
    if (t + u < KT) step(u, t + u);                        // (uniform over the workgroup)
#pragma unroll
  for (int j = 0; j < FN; ++j)
    if (p.partial)
      store_partial(p, acc[j], blockIdx.y, m0 + xrow - r, n0 + wrow[j], lane);
    else
      store_frag<_Float16>(p, acc[j], m0 + xrow - r, n0 + wrow[j], lane);
}

// ---------------------------------------------------------------- tiles loaded straight into LDS
// (32 FM) x (64 NCG) tile, NCG x KG waves, k tiles of BK in NST LDS stages.
//
// Staged as in the kernel above, every byte passes through registers and a ds_write on its way into
// LDS, the widened weights are twice their bytes there and are read once per row of waves.  Here
//  * both operands are loaded into LDS as they are in memory (buffer_load ... lds), NST - 1 tiles
//    ahead: nothing waits in registers;
//  * a wave multiplies all rows of the tile with 64 output channels, and its KG'th of every k
//    tile: each weight byte is read from LDS by one wave only, as a byte, and widened once;
//  * what a wave issues next to its MFMAs decides (a vector instruction of either of a SIMD's two
//    waves runs next to an MFMA only while that is past its operand reads: about 3.5 of them per
//    MFMA are free, the others add to it): widening is 16 instructions per 64 channels x 16 of k,
//    shared by the 2 FM MFMAs that use them -- hence wave tiles of 128 rows where there are that
//    many --, addresses advance in scalar registers, and reads, loads and widening are dealt out
//    over the MFMAs.  Sent out together behind the barrier, the loads of all waves queue at the
//    compute unit's address path (25 clocks apiece), the reads at the LDS, and every wave's MFMAs
//    behind them;
//  * a wave takes one 32-deep unit of every k tile (BK = 32 KG), and there is one barrier per k tile, in the
//    middle of it: by then all fragments of the tile are in registers, its stage takes the tile NST
//    further on, and the next tile's fragments are read under the unit's second half.
// The sums of the k groups meet in LDS at the end, which also puts the results into whole rows.
// f32 activations stay f32 in LDS; a wave splits the fragments it reads (hi = half(x), lo = half(x
// - hi)) and multiplies both.
// LDS blocks as in the int8 kernels: 8 rows x 128 bytes, chunk c of row r in slot c ^ r ^ (block &
// 1): whole lines for the loads, all banks for the fragment reads.
// Against the staged kernel, f16: 1024 x 4096 -> 4096 42.9 -> 34.8 us (power: 24.6 on constant operands),
// 256 x 4096 -> 11008 36.3 -> 28.0, 64 x 4096 -> 4096 13.5 -> 11.9, 290 x 1600 -> 752 10.5 -> 7.2, 4096^3
// 133 -> 124; f32: 128 x 4096 -> 4096 23.1 -> 16.2, 1024 x 2048 -> 2048 31.6 -> 23.8, 1549 x 2208 -> 5628
// 125 -> 95.5.
template <typename XT, int FM, int NCG, int KG, int BK, int NST>
struct DmaShape {
  static constexpr int kBM = 32 * FM, kBN = 64 * NCG, kWaves = NCG * KG;
  static constexpr int kStage = (kBM * (int)sizeof(XT) + kBN) * BK;
  // the epilogue's sums: 64 rows (32 where the tile has no more) of every k group, rows padded by
  // 16 bytes so that a fragment's writes spread over the banks
  static constexpr int kPitch = kBN + 4, kRows = FM > 1 ? 64 : 32;
  static constexpr int kSums = KG * kRows * kPitch * 4;
  static constexpr int kTiles = NST * kStage > kSums ? NST * kStage : kSums;
  // behind them: zero points (64 per wave), then the scale and the bias of every channel
  static constexpr int kZp = kTiles, kFactors = kZp + kWaves * 256, kLds = kFactors + kBN * 8;
};

template <typename XT, bool SIGNED, int FM, int NCG, int KG, int BK, int NST, bool WORDS>
__global__ void __launch_bounds__(NCG* KG * 64, 2) wo_dma_kernel(const WoParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  using Shape = DmaShape<XT, FM, NCG, KG, BK, NST>;
  constexpr bool F32 = sizeof(XT) == 4;
  constexpr int BM = Shape::kBM, BN = Shape::kBN, NW = Shape::kWaves;
  constexpr int SUBS = BK * (int)sizeof(XT) / 128;       // 128-byte wide pieces of an activation row's k tile
  constexpr int WR = 1024 / BK;                          // weight rows per load
  constexpr int A_LD = SUBS * (BM / 8) / NW, W_LD = (BN / WR) / NW, LD = A_LD + W_LD;
  constexpr int A_BYTES = BM * 128 * SUBS, STAGE = Shape::kStage;
  constexpr int CH = F32 ? 2 : 1;                        // 16-byte chunks of an activation row per 16 of k and lane
  constexpr unsigned kFlip = SIGNED ? 0x80808080u : 0u;
  constexpr int kPast = (int)0x80000000;                 // an offset no descriptor covers
  static_assert((BK == 64 || BK == 128) && BK == 32 * KG, "a wave takes one 32-deep unit of a k tile");
  static_assert(STAGE == A_BYTES + BN * BK && Shape::kLds <= 160 * 1024, "LDS");
  static_assert((SUBS * (BM / 8)) % NW == 0 && (BM / 8) % 2 == 0 && NW % 2 == 0, "loads of a wave");
  static_assert((BN / WR) % NW == 0 && NST * LD <= 63, "loads of a wave; vmcnt is a 6-bit counter");
  extern __shared__ __attribute__((aligned(1024))) uint8_t wo_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cg = wave % NCG, kg = wave / NCG;
  const int r = lane & 31, g = lane >> 5;

  // Workgroups go to the 8 XCDs in turn, and each has its own L2: an XCD takes a contiguous range
  // of tiles, walked in panels of 512 rows, so that what it has running at a time shares rows of
  // both operands.
  const int tiles_n = (p.N + BN - 1) / BN, tiles_m = (p.M + BM - 1) / BM;
  int tile = blockIdx.x;
  {
    const int tiles = gridDim.x, q = tiles >> 3, rem = tiles & 7, x = tile & 7;
    tile = x * q + min(x, rem) + (tile >> 3);
  }
  const int panel_rows = min(tiles_m, 512 / BM);
  const int panel = tile / (panel_rows * tiles_n), in_panel = tile - panel * panel_rows * tiles_n;
  const int rows_here = min(panel_rows, tiles_m - panel * panel_rows);
  const int m0 = (panel * panel_rows + in_panel % rows_here) * BM, n0 = (in_panel / rows_here) * BN;
  const int kbeg = blockIdx.y * p.k_split;               // this workgroup's k range
  const int klen = min(p.K, kbeg + p.k_split) - kbeg;
  const int KT = (klen + BK - 1) / BK;
  // descriptors over the tile's rows from (first row, kbeg) on, moved on with the tiles that are
  // loaded; the host has checked that the offsets below fit 31 bits
  const int mrows = min(BM, p.M - m0), nrows = min(BN, p.N - n0);
  const XT* xbase = static_cast<const XT*>(p.x) + (int64_t)m0 * p.ldx + kbeg;
  const uint8_t* wbase = p.w + (int64_t)n0 * p.w_sn + kbeg;
  const int xbytes = (int)(((int64_t)(mrows - 1) * p.ldx + klen) * (int)sizeof(XT));
  const int wbytes = (int)((int64_t)(nrows - 1) * p.w_sn + klen);
  const unsigned lds_base =
      (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(size_t)(lds_void_t*)wo_lds);

  // ---- loads.  Load q = wave + i NW of the workgroup fills 1 KiB block q: 8 rows x 128 bytes,
  // lane -> row lane / 8, slot lane % 8.  The number of waves is even, so the parity of a block is
  // the wave's and a lane takes the same chunk of a row in all its loads.
  const int lr = lane >> 3;
  const int ck = ((lane & 7) ^ lr ^ (wave & 1)) << 4;    // byte offset of that chunk
  // (weight rows of 64 bytes: 16 to a block, chunk c of row r in slot c ^ (r / 4 & 3))
  const int cw = BK == 128 ? ck : ((lane & 3) ^ (lane >> 4)) << 4;
  int xo[A_LD], wo[W_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) {
    const int q = wave + i * NW, row = (q % (BM / 8)) * 8 + lr;
    // (rows past the last: zeros, no memory touched)
    xo[i] = row < mrows ? (int)(row * p.ldx * (int)sizeof(XT)) + q / (BM / 8) * 128 + ck : kPast;
  }
#pragma unroll
  for (int i = 0; i < W_LD; ++i) {
    const int row = (wave + i * NW) * WR + lane / (BK / 16);
    wo[i] = row < nrows ? (int)(row * p.w_sn) + cw : kPast;
  }
  // load l of tile t; FULL: the tile is whole (otherwise zeros past the range's end; K % 16 == 0 but with WORDS).
  // WORDS: rows that begin on four bytes, K % 4 == 0.  A group of 16 k that holds the end of the range is loaded as the
  // 16 in front of that end, of both operands (no load leaves its row), and the activations that the group before holds
  // already are made zero where they are multiplied.  The descriptors of such tiles begin 16 k earlier, so
  // that no offset is negative.  (In one kernel with the aligned rows' form those took 7.6 in place of 7.05 us at 64 x
  // 2048 -> 1000.)
  auto issue_load = [&](auto full_c, auto l_c, int t, int st) {
    constexpr bool FULL = decltype(full_c)::value != 0;
    constexpr int l = decltype(l_c)::value;
    const int k0 = t * BK;
    const unsigned base = lds_base + st * STAGE + wave * 1024;
    if constexpr (l < A_LD) {
      const int first = ((wave + l * NW) / (BM / 8) * 128 + ck) / (int)sizeof(XT);   // the chunk's first element in the tile
      if constexpr (FULL || !WORDS) {
        const v4i rs = make_rsrc(xbase + k0, xbytes - k0 * (int)sizeof(XT));
        buffer_load_lds_b128(rs, base + l * NW * 1024, FULL || k0 + first < klen ? xo[l] : kPast);
      } else {
        const v4i rs = make_rsrc(xbase + k0 - 16, xbytes - (k0 - 16) * (int)sizeof(XT));
        const int left = klen - k0 - (first & ~15);
        buffer_load_lds_b128(rs, base + l * NW * 1024, left > 0 ? xo[l] + min(left, 16) * (int)sizeof(XT) : kPast);
      }
    } else {
      constexpr int at = A_BYTES + (l - A_LD) * NW * 1024;
      if constexpr (FULL || !WORDS) {
        buffer_load_lds_b128(make_rsrc(wbase + k0, wbytes - k0), base + at, FULL || k0 + cw < klen ? wo[l - A_LD] : kPast);
      } else {
        const int left = klen - k0 - cw;
        buffer_load_lds_b128(make_rsrc(wbase + k0 - 16, wbytes - (k0 - 16)), base + at,
                             left > 0 ? wo[l - A_LD] + min(left, 16) : kPast);
      }
    }
  };

  // ---- fragments: row r of a 32-row block, 16 values of k from 16 g of a 32-deep unit on
  const int swz = (r & 7) ^ ((r >> 3) & 1);
  const int row_off = (r >> 3) * 1024 + (r & 7) * 128;
  int a_off[2 * CH];
  {
    const int sub = F32 ? kg : kg >> 1, first = F32 ? 4 * g : 4 * (kg & 1) + 2 * g;
#pragma unroll
    for (int h = 0; h < 2 * CH; ++h) a_off[h] = sub * BM * 128 + row_off + (((first + h) ^ swz) << 4);
  }
  const int w_off = A_BYTES + cg * 64 * BK + (BK == 128 ? row_off + (((2 * kg + g) ^ swz) << 4)
                                                        : r * 64 + (((2 * kg + g) ^ ((r >> 2) & 3)) << 4));
  h2 c[2];
  u4 fa[2][FM][CH];                  // activations of the unit's two 16-deep steps
  u4 fw[2][2];                       // weights of this k tile and the next: both steps
  h8 w[2][2];                        // widened: of this step and the next
  // read q of a unit's fragments: the weights, then the activations of row block (q - 2) / (2 CH)
  constexpr int READS = 2 + FM * 2 * CH;
  auto read = [&](auto set_c, auto q_c, const uint8_t* base) {
    constexpr int set = decltype(set_c)::value, q = decltype(q_c)::value;
    if constexpr (q < 2) {
      fw[set][q] = *reinterpret_cast<const u4*>(base + w_off + q * 32 * BK);
    } else {
      constexpr int i = (q - 2) / (2 * CH), h = (q - 2) % (2 * CH);
      fa[h / CH][i][h % CH] = *reinterpret_cast<const u4*>(base + a_off[h] + i * 4096);
    }
  };
  auto widen = [&](auto set_c, auto s_c, int j) {
    constexpr int set = decltype(set_c)::value, s = decltype(s_c)::value;
    w[s][j] = widen8(fw[set][j][2 * s], fw[set][j][2 * s + 1], kFlip, c[j]);
  };
  // (the low halves' products, 2^-11 of the others, on sums of their own: half the roundings at the
  // size of the whole sum, 0.67 of the rms error against 64 bits that one sum for both gives)
  f16v acc[FM][2], acc_lo[F32 ? FM : 1][2];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[i][j][v] = 0.0f;
        acc_lo[F32 ? i : 0][j][v] = 0.0f;
      }
  // One 16-deep step, a row block (two MFMAs per part) at a time, behind each of them hook(i) and a
  // share of the widening of the next step's weights (of set `next`).
  auto step = [&](auto s_c, auto next_c, auto&& hook) {
    constexpr int s = decltype(s_c)::value;
    static_for_n<FM>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      h8 a[F32 ? 2 : 1];
      if constexpr (F32) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const f4 v = __builtin_bit_cast(f4, fa[s][i][e / 4 % CH]);
          h2 hi, lo;
          split2(v[e % 4], v[e % 4 + 1], hi, lo);
          a[0][e] = hi.x, a[0][e + 1] = hi.y;
          a[1][e] = lo.x, a[1][e + 1] = lo.y;
        }
      } else {
        a[0] = __builtin_bit_cast(h8, fa[s][i][0]);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[s][j], a[0], acc[i][j], 0, 0, 0);
      if constexpr (F32) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc_lo[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[s][j], a[1], acc_lo[i][j], 0, 0, 0);
      }
      hook(i_c);
      if constexpr (i == (FM > 1 ? FM - 2 : 0)) widen(next_c, Int<s ^ 1>(), 0);
      if constexpr (i == FM - 1) widen(next_c, Int<s ^ 1>(), 1);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // until tile t has landed: at most the tiles behind it of those issued so far are in flight
  auto landed = [&](int behind) {
    static_for_n<NST>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      if (behind == k) __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(k * LD));
    });
  };

  // Scale and bias of channel tid, and the zero points of the wave's channels, ahead of the tiles: a
  // use of a value loaded the ordinary way waits for every load before it, so the first are not
  // touched until the end and the second go through LDS like the tiles.
  // (As bits, and from the scales' place where there is no bias: nothing to be done to them here.)
  using Raw = std::conditional_t<F32, uint32_t, uint16_t>;
  const int own = n0 + min(tid, nrows - 1);
  const Raw raw_s = static_cast<const Raw*>(p.scale)[own];
  const Raw raw_b = static_cast<const Raw*>(p.bias ? p.bias : p.scale)[own];
  if (p.zp)
    buffer_load_lds_b32(make_rsrc(p.zp + n0, (int64_t)nrows * 4), lds_base + Shape::kZp + wave * 256, (cg * 64 + lane) * 4);
  static_for_n<NST>([&](auto t_c) {
    constexpr int t = decltype(t_c)::value;
    if (t < KT) static_for_n<LD>([&](auto l_c) { issue_load(Int<0>(), l_c, t, t); });
  });
  landed(min(KT, NST) - 1);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int zp = p.zp ? *reinterpret_cast<const int*>(wo_lds + Shape::kZp + wave * 256 + (j * 32 + r) * 4) : 0;
    const _Float16 v = (_Float16)(float)(1024 + zp + (SIGNED ? 128 : 0));
    c[j] = (h2){v, v};
  }
  static_for_n<READS>([&](auto q_c) { read(Int<0>(), q_c, wo_lds); });
  widen(Int<0>(), Int<0>(), 0);
  widen(Int<0>(), Int<0>(), 1);

  // Tile t's stage is free from its middle on and takes tile t + NST, whose loads are dealt out from
  // there to the middle of tile t + 1: over this tile's second step (SLOT 0 on) and the next one's first.
  auto spread = [&](auto count_c, auto slots_c, auto slot_c, auto&& body) {
    constexpr int count = decltype(count_c)::value, slots = decltype(slots_c)::value, slot = decltype(slot_c)::value;
    static_for_n<count>([&](auto l_c) {
      if constexpr (decltype(l_c)::value * slots / count == slot) body(l_c);
    });
  };
  constexpr int SLOTS = 2 * FM;
  int st = 0;                                            // tile t's stage
  // one k tile; PAR: the set its weights are in; MORE: the tiles loaded meanwhile are there, and whole
  auto k_tile = [&](auto more_c, auto par_c, int t) {
    constexpr int MORE = decltype(more_c)::value, PAR = decltype(par_c)::value;
    using Next = Int<PAR ^ 1>;
    const int pst = st == 0 ? NST - 1 : st - 1, nst = st + 1 == NST ? 0 : st + 1;
    const uint8_t* there = wo_lds + nst * STAGE;
    const bool next = MORE || t + 1 < KT;                // (uniform)
    if constexpr (WORDS && !MORE) {
      static_assert(!F32, "f32 rows on four bytes: wo_exact_f32_kernel");
      if ((klen & 15) != 0 && t == KT - 1) {             // (uniform) the words that came twice
        const int left = klen - t * BK - 32 * kg - 16 * g;
        const int twice = left > 0 ? max(16 - left, 0) : 0;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          fa[0][i][0] = zero_first(fa[0][i][0], min(twice, 8));
          fa[1][i][0] = zero_first(fa[1][i][0], max(twice - 8, 0));
        }
      }
    }
    step(Int<0>(), Int<PAR>(), [&](auto i_c) {
      if (MORE || (t > 0 && t - 1 + NST < KT))
        spread(Int<LD>(), Int<SLOTS>(), Int<FM + decltype(i_c)::value>(),
               [&](auto l_c) { issue_load(Int<MORE>(), l_c, t - 1 + NST, pst); });
    });
    if (next) {
      if constexpr (MORE)
        __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((NST - 2) * LD));
      else
        landed(min(KT - 2 - t, NST - 2));
      __syncthreads();                                   // tile t + 1 is in LDS; tile t is in registers
    }
    __builtin_amdgcn_sched_barrier(0);
    step(Int<1>(), Next(), [&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      // the next tile's fragments: the weights ahead of the others, a row block's activations behind
      // its MFMAs, in their registers
      if (next)
        static_for_n<READS>([&](auto q_c) {
          constexpr int q = decltype(q_c)::value;
          if constexpr (q < 2 ? i == 0 : (q - 2) / (2 * CH) == i) read(Next(), q_c, there);
        });
      if (MORE || t + NST < KT)
        spread(Int<LD>(), Int<SLOTS>(), i_c, [&](auto l_c) { issue_load(Int<MORE>(), l_c, t + NST, st); });
    });
    st = nst;
  };
  // (the first step has no loads left over from one before it; then those whose loads are whole tiles;
  // then the others)
  const int whole = klen / BK - NST;
  k_tile(Int<0>(), Int<0>(), 0);
  int t = 1;
  for (; t + 1 < whole; t += 2) {
    k_tile(Int<1>(), Int<1>(), t);
    k_tile(Int<1>(), Int<0>(), t + 1);
  }
  for (; t + 1 < KT; t += 2) {
    k_tile(Int<0>(), Int<1>(), t);
    k_tile(Int<0>(), Int<0>(), t + 1);
  }
  if (t < KT) k_tile(Int<0>(), Int<1>(), t);

  if constexpr (F32) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] += acc_lo[i][j];
  }
  // ---- the k groups' sums into LDS, 64 rows at a time, and out as rows: lane (r, g) holds of a
  // fragment row r, channels 8 q + 4 g .. + 3
  constexpr int P = Shape::kPitch, ROWS = Shape::kRows;
  constexpr int CPR = BN / 8, RPP = NW * 64 / CPR;       // threads (8 channels each) per row, rows per pass
  float* const sums = reinterpret_cast<float*>(wo_lds);
  float* const factors = reinterpret_cast<float*>(wo_lds + Shape::kFactors);
  const int n = n0 + (tid % CPR) * 8;
  if (tid < BN) {
    factors[tid] = to_f32(__builtin_bit_cast(XT, raw_s));
    factors[BN + tid] = p.bias ? to_f32(__builtin_bit_cast(XT, raw_b)) : 0.0f;
  }
  float sc[8], bi[8];
  // (16-byte pieces of any alignment: rows of N elements need not be multiples of 16 bytes)
  typedef _Float16 h8_any __attribute__((ext_vector_type(8), aligned(2)));
  typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));
  const bool whole8 = n + 8 <= p.N;
  static_for_n<(FM + 1) / 2>([&](auto h_c) {
    constexpr int h = decltype(h_c)::value;
    __syncthreads();                                     // the stages, or the rows before, have been read
#pragma unroll
    for (int i = 0; i < ROWS / 32; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<f4*>(&sums[(kg * ROWS + i * 32 + r) * P + cg * 64 + j * 32 + 8 * q + 4 * g]) =
              (f4){acc[2 * h + i][j][4 * q], acc[2 * h + i][j][4 * q + 1], acc[2 * h + i][j][4 * q + 2],
                   acc[2 * h + i][j][4 * q + 3]};
    __syncthreads();
    if (h == 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        sc[e] = factors[(tid % CPR) * 8 + e];
        bi[e] = factors[BN + (tid % CPR) * 8 + e];
      }
    }
#pragma unroll
    for (int pass = 0; pass < ROWS / RPP; ++pass) {
      const int row = tid / CPR + pass * RPP, m = m0 + 64 * h + row;
      float s[8];
#pragma unroll
      for (int k = 0; k < KG; ++k) {
        const f4* src = reinterpret_cast<const f4*>(&sums[(k * ROWS + row) * P + (tid % CPR) * 8]);
        const f4 lo = src[0], hi = src[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[e] = k ? s[e] + lo[e] : lo[e];
          s[4 + e] = k ? s[4 + e] + hi[e] : hi[e];
        }
      }
      if (m >= p.M || n >= p.N) continue;
      if (p.partial) {
        float* dst = p.partial + ((int64_t)blockIdx.y * p.M + m) * p.N + n;
        if (whole8) {
          *reinterpret_cast<f4_any*>(dst) = (f4){s[0], s[1], s[2], s[3]};
          *reinterpret_cast<f4_any*>(dst + 4) = (f4){s[4], s[5], s[6], s[7]};
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n + e < p.N) dst[e] = s[e];
        }
        continue;
      }
      XT* dst = static_cast<XT*>(p.out) + (int64_t)m * p.ldo + n;
      XT y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = (XT)(s[e] * sc[e] + bi[e]);
      if (whole8) {
        if constexpr (F32) {
          *reinterpret_cast<f4_any*>(dst) = (f4){y[0], y[1], y[2], y[3]};
          *reinterpret_cast<f4_any*>(dst + 4) = (f4){y[4], y[5], y[6], y[7]};
        } else {
          *reinterpret_cast<h8_any*>(dst) = (h8){y[0], y[1], y[2], y[3], y[4], y[5], y[6], y[7]};
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (n + e < p.N) dst[e] = y[e];
      }
    }
  });
#else
  (void)p;
#endif
}

// out = (sum over the k ranges, in their order) * scale + bias: the second half of a split
// launch.  VEC consecutive channels per thread.
template <typename XT, int VEC>
__global__ void __launch_bounds__(256) wo_splitk_reduce_kernel(const WoParams p, int splits) {
  const int nv = p.N / VEC;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)p.M * nv) return;
  const int m = (int)(idx / nv), n = (int)(idx % nv) * VEC;
  const int64_t plane = (int64_t)p.M * p.N;
  const float* src = p.partial + (int64_t)m * p.N + n;
  float sum[VEC];
  if constexpr (VEC == 4) {
    f4 v = *reinterpret_cast<const f4*>(src);
    for (int s = 1; s < splits; ++s) v += *reinterpret_cast<const f4*>(src + s * plane);
    sum[0] = v.x, sum[1] = v.y, sum[2] = v.z, sum[3] = v.w;
  } else {
    sum[0] = src[0];
    for (int s = 1; s < splits; ++s) sum[0] += src[s * plane];
  }
  const XT* scale = static_cast<const XT*>(p.scale);
  const XT* bias = static_cast<const XT*>(p.bias);
  XT* out = static_cast<XT*>(p.out) + (int64_t)m * p.ldo + n;
#pragma unroll
  for (int e = 0; e < VEC; ++e)
    out[e] = (XT)(sum[e] * to_f32(scale[n + e]) + (bias ? to_f32(bias[n + e]) : 0.0f));
}

// ---------------------------------------------------------------- small-M kernel, M <= 32 MT
// MT blocks of 32 rows against 32 output channels per workgroup: the weights of those
// channels are read once, whatever M.
template <typename XT, int NW, int MT>
__global__ void __launch_bounds__(NW * 64) wo_skinny_kernel(const WoParams p) {
  __shared__ float red[NW - 1][16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, g = lane >> 5;
  const int n0 = blockIdx.x * 32;
  const int n = min(n0 + r, p.N - 1);
  const XT* xrow[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    xrow[i] = static_cast<const XT*>(p.x) + (int64_t)min(i * 32 + r, p.M - 1) * p.ldx + 16 * g;
  const uint8_t* wrow = p.w + (int64_t)n * p.w_sn + 16 * g;
  const h2 c = centre(p, n);
  f16v acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;
  const u4 zero = {0, 0, 0, 0};
  // chunks of 32 dealt round-robin over the waves, U in flight per wave: with one byte per
  // weight from HBM the kernel lives on the bytes it keeps in flight
  constexpr int U = MT == 1 ? 4 : (MT == 4 && sizeof(XT) == 4 ? 1 : 2);   // (register budget)
  for (int k0 = wave * 32; k0 < p.K; k0 += U * NW * 32) {
    XFrag<XT> xf[U][MT];
    u4 wf[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = k0 + u * NW * 32;
      const bool valid = kk + 16 * g < p.K;
      const int k = valid ? kk : 0;
      wf[u] = valid ? *reinterpret_cast<const u4*>(wrow + k) : zero;
#pragma unroll
      for (int i = 0; i < MT; ++i) xf[u][i].load(xrow[i] + k, valid);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      h8 w0, w1;
      widen16(wf[u], p.flip, c, w0, w1);
#pragma unroll
      for (int part = 0; part < XFrag<XT>::kParts; ++part)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[u][i].step(part, 0), w0, acc[i], 0, 0,
                                                          0);
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[u][i].step(part, 1), w1, acc[i], 0, 0,
                                                          0);
        }
    }
  }
  // partial sums of the waves, one row block at a time through the same 28 KiB of LDS
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (i > 0) __syncthreads();
    if (wave > 0) {
#pragma unroll
      for (int v = 0; v < 16; ++v) red[wave - 1][v][lane] = acc[i][v];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int w = 1; w < NW; ++w)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][v] += red[w - 1][v][lane];
      store_frag<XT>(p, acc[i], i * 32, n0 + r, lane);
    }
  }
}

// ---------------------------------------------------------------- M <= 2: matrix times one or two vectors
// One wave per output channel streams that channel's weight row from end to end -- 64 lanes x
// 16 bytes = 1 KiB contiguous per load instruction, U of them in flight -- and multiplies it
// with the activation rows, which the workgroup keeps in LDS (f32 ones as hi and lo halves),
// on the vector ALUs (v_dot2_f32_f16: the matrix cores have nothing to gain on one or two
// rows, and a row read linearly keeps one DRAM page open where 16 rows read side by side keep
// 16).  The lanes' partial sums meet in a butterfly of cross-lane shuffles.
template <typename XT, int NW, int MR, int U>
__global__ void __launch_bounds__(NW * 64) wo_gemv_kernel(const WoParams p) {
  constexpr bool F32 = sizeof(XT) == 4;
  extern __shared__ __attribute__((aligned(16))) uint8_t wo_lds[];   // [MR][hi | lo][K] halves
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = blockIdx.x * NW + __builtin_amdgcn_readfirstlane(wave);
  const int kpad = (p.K + 7) & ~7;                       // (K % 16 == 0 anyway)
  // the activation rows into LDS, 8 elements per thread and step
  for (int i = threadIdx.x; i < MR * (kpad >> 3); i += NW * 64) {
    const int m = i / (kpad >> 3), k = (i - m * (kpad >> 3)) << 3;
    const XT* src = static_cast<const XT*>(p.x) + (int64_t)min(m, p.M - 1) * p.ldx + k;
    h8 hi, lo;
    if constexpr (F32) {
      const f4 a = *reinterpret_cast<const f4*>(src), b = *reinterpret_cast<const f4*>(src + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = e < 4 ? a[e] : b[e - 4];
        hi[e] = (_Float16)v;
        lo[e] = (_Float16)(v - (float)hi[e]);
      }
      *reinterpret_cast<h8*>(&wo_lds[((2 * m + 1) * kpad + k) * 2]) = lo;
      *reinterpret_cast<h8*>(&wo_lds[((2 * m) * kpad + k) * 2]) = hi;
    } else {
      *reinterpret_cast<h8*>(&wo_lds[(m * kpad + k) * 2]) = *reinterpret_cast<const h8*>(src);
    }
  }
  __syncthreads();
  if (n >= p.N) return;                                  // (no barrier below)
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.w + (int64_t)n * p.w_sn), 0, p.K, kBufferRsrcWord3);
  const h2 c = centre(p, n);
  float acc[MR];
#pragma unroll
  for (int m = 0; m < MR; ++m) acc[m] = 0.0f;
  for (int k0 = 16 * lane; k0 < p.K; k0 += U * 1024) {
    u4 wq[U];
#pragma unroll
    for (int u = 0; u < U; ++u)                          // (past K: zeros, no memory touched)
      wq[u] = __builtin_amdgcn_raw_buffer_load_b128(wrs, k0 + u * 1024, 0, 0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * 1024;
      if (k < p.K) {
        h8 w0, w1;
        widen16(wq[u], p.flip, c, w0, w1);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
#pragma unroll
          for (int part = 0; part < (F32 ? 2 : 1); ++part) {
            const uint8_t* xs = &wo_lds[(((F32 ? 2 * m + part : m) * kpad) + k) * 2];
            const h8 x0 = *reinterpret_cast<const h8*>(xs), x1 = *reinterpret_cast<const h8*>(xs + 16);
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
              acc[m] = __builtin_amdgcn_fdot2((h2){x0[e], x0[e + 1]}, (h2){w0[e], w0[e + 1]}, acc[m], false);
              acc[m] = __builtin_amdgcn_fdot2((h2){x1[e], x1[e + 1]}, (h2){w1[e], w1[e + 1]}, acc[m], false);
            }
          }
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    float v = acc[m];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane == 0 && m < p.M) {
      const float sc = to_f32(static_cast<const XT*>(p.scale)[n]);
      const float b = p.bias ? to_f32(static_cast<const XT*>(p.bias)[n]) : 0.0f;
      static_cast<XT*>(p.out)[(int64_t)m * p.ldo + n] = (XT)(v * sc + b);
    }
  }
}

typedef float f4v __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- up to 32 rows, operands through LDS
// 16 MT rows x 16 FN output channels per workgroup on v_mfma_f32_16x16x32_f16, the k range dealt
// over the waves in units of 64.  Bound by the weight bytes from HBM.  When every lane fetches its
// own activation row (wo_skinny_kernel: 32 rows x 32 bytes per load instruction), the compute
// unit's address path, not HBM, sets the pace from nine rows on.  Here a wave loads each unit the
// way memory likes it -- eight lanes (sixteen for f32) per 128-byte (256-byte) row segment of the
// activations, four per 64-byte segment of the weights --, keeps D units in registers on their way
// from memory, and turns them into MFMA fragments through a piece of LDS that only this wave touches
// (no barrier: the LDS executes a wave's instructions in order).  f32 activations are split into hi
// and lo half tiles there.
// The width is what balances the chip: with 32 channels and 32 rows per workgroup in every case,
// 11008 channels were 344 workgroups on 256 compute units, one at a time in 144 registers, and half
// the multiplications met rows that were not there.  4096 -> 11008, M = 16: f16 14.6 -> 11.3 us (18.3 ->
// 13.9 with weights from HBM, 3.2 TB/s), f32 21.5 -> 12.7; 8192 -> 2048 11.3 -> 7.9; M = 32, 4096 -> 11008
// 18.8 -> 12.1.  More units in registers were slower (D = 4 in place of 2: M = 32 14.0, f32 14.5)
// except for the narrowest form (4096 -> 8192 9.5 against 10.6).
// RAGGED (f16): as in wo_ragged_kernel (M = 16, 3001 -> 4096, one output per thread before: 567 us).
constexpr int kRowsWaves = 8;

template <typename XT, int MT, int FN, int D, bool RAGGED = false>
__global__ void __launch_bounds__(kRowsWaves * 64) wo_rows_kernel(const WoParams p) {
  constexpr bool F32 = sizeof(XT) == 4;
  static_assert(!RAGGED || !F32, "f32 activations: wo_exact_f32_kernel");
  constexpr int NW = kRowsWaves, MR = 16 * MT, BN = 16 * FN;
  constexpr int XL = F32 ? 16 : 8;                       // lanes per activation row of a unit
  constexpr int XP = MR * XL / 64;                       // activation loads per lane and unit
  constexpr int XBYTES = MR * 128 * (F32 ? 2 : 1);       // [hi, then lo] half tiles
  constexpr int WBYTES = BN * 64;
  static_assert(D * (XP + FN) <= 63, "vmcnt is a 6-bit counter");
  static_assert(MT * FN <= NW && MT * FN * 1024 <= XBYTES + WBYTES, "the waves' partial sums fit the LDS");
  extern __shared__ __attribute__((aligned(16))) uint8_t wo_lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * BN;
  const int nrows = min(BN, p.N - n0), mrows = min(MR, p.M);
  uint8_t* const xs = wo_lds + wave * (XBYTES + WBYTES);
  uint8_t* const ws = xs + XBYTES;
  // descriptors over the activation rows and this workgroup's weight rows; the host has
  // checked that the byte offsets fit 31 bits
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(p.x), 0, (int)(((int64_t)(mrows - 1) * p.ldx + p.K) * sizeof(XT)),
      kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.w + (int64_t)n0 * p.w_sn), 0,
      (int)((int64_t)(nrows - 1) * p.w_sn + p.K), kBufferRsrcWord3);
  constexpr int kPast = (int)0x80000000;                 // an offset no descriptor covers

  // global -> LDS assignment
  const int xc = lane & (XL - 1), wc = lane & 3;
  int xo[XP], xl[XP];
  bool xok[XP];
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int row = lane / XL + (64 / XL) * i;
    const int sx = (row ^ (row >> 3)) & 7;
    xok[i] = row < mrows;                                // (rows past M are never stored)
    xo[i] = (int)((int64_t)min(row, mrows - 1) * p.ldx * sizeof(XT)) + (RAGGED ? 0 : 16 * xc);
    xl[i] = F32 ? row * 128 + (((xc >> 1) ^ sx) << 4) + 8 * (xc & 1)
                : row * 128 + ((xc ^ sx) << 4);
  }
  int wo[FN], wl[FN];
#pragma unroll
  for (int i = 0; i < FN; ++i) {
    const int row = (lane >> 2) + 16 * i;
    wo[i] = (int)((int64_t)min(row, nrows - 1) * p.w_sn) + (RAGGED ? 0 : 16 * wc);
    wl[i] = row * 64 + ((wc ^ ((row >> 2) & 3)) << 4);
  }
  h2 c[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) c[j] = centre(p, n0 + min(16 * j + r, nrows - 1));
  u4 xr[D][XP], wr[D][FN];
  const uint8_t* xbase = static_cast<const uint8_t*>(p.x);
  const uint8_t* wbase = p.w + (int64_t)n0 * p.w_sn;
  auto fetch = [&](u4* xq, u4* wq, int k0) {
    if constexpr (RAGGED) {
      const unsigned kx = min(k0 + 16 * (xc >> 1), p.K - 16) + 8 * (xc & 1);
      const unsigned kw = min(k0 + 16 * wc, p.K - 16);
#pragma unroll
      for (int i = 0; i < XP; ++i) xq[i] = load_any(xbase, (unsigned)xo[i] + 2 * kx);
#pragma unroll
      for (int i = 0; i < FN; ++i) wq[i] = load_any(wbase, (unsigned)wo[i] + kw);
      return;
    }
    const bool xv = k0 + (F32 ? 4 : 8) * xc < p.K, wv = k0 + 16 * wc < p.K;   // K % 16 == 0
#pragma unroll
    for (int i = 0; i < XP; ++i)
      xq[i] = __builtin_amdgcn_raw_buffer_load_b128(
          xrs, xv && xok[i] ? xo[i] + (int)sizeof(XT) * k0 : kPast, 0, 0);
#pragma unroll
    for (int i = 0; i < FN; ++i)
      wq[i] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wv ? wo[i] + k0 : kPast, 0, 0);
  };
  auto park = [&](u4* xq, const u4* wq, int k0) {
    if (RAGGED && k0 + 64 > p.K) {                         // (uniform) the end of the rows
      const int c16 = k0 + 16 * (xc >> 1);
      const int z = c16 - min(c16, p.K - 16) - 8 * (xc & 1);
#pragma unroll
      for (int i = 0; i < XP; ++i) xq[i] = zero_first(xq[i], z);
    }
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      if constexpr (F32) {
        const f4 v = __builtin_bit_cast(f4, xq[i]);
        h2 hi[2], lo[2];
        split2(v[0], v[1], hi[0], lo[0]);
        split2(v[2], v[3], hi[1], lo[1]);
        *reinterpret_cast<h4*>(&xs[xl[i]]) = (h4){hi[0].x, hi[0].y, hi[1].x, hi[1].y};
        *reinterpret_cast<h4*>(&xs[MR * 128 + xl[i]]) = (h4){lo[0].x, lo[0].y, lo[1].x, lo[1].y};
      } else {
        *reinterpret_cast<u4*>(&xs[xl[i]]) = xq[i];
      }
    }
#pragma unroll
    for (int i = 0; i < FN; ++i) *reinterpret_cast<u4*>(&ws[wl[i]]) = wq[i];
  };
  // f32, more than 16 rows and channels: the low halves' products on sums of their own, as in wo_dma_kernel,
  // and the waves' sums added in pairs: 0.65-0.78 of the rms error against 64 bits of one sum added wave by
  // wave, for 0-2 % of the time (1024 of k 0.87e-7 against 1.25e-7, tiles 0.96e-7; 2048 1.00e-7 / 1.53e-7 /
  // 1.21e-7).  Up to 16 rows the registers would cost a compute unit its second workgroup.
  constexpr bool kLowSums = F32 && MT == 2 && FN > 1;
  f4v acc[MT][FN], acc_lo[kLowSums ? MT : 1][FN];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      acc[i][j] = (f4v){0.f, 0.f, 0.f, 0.f};
      acc_lo[kLowSums ? i : 0][j] = (f4v){0.f, 0.f, 0.f, 0.f};
    }
  // lane (r, g): the unit's k values 16 g .. 16 g + 15 of row r of a fragment, as two k steps
  auto multiply = [&]() {
    h8 a[F32 ? 2 : 1][MT][2];
#pragma unroll
    for (int part = 0; part < (F32 ? 2 : 1); ++part)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int row = 16 * i + r, sx = (row ^ (row >> 3)) & 7;
          a[part][i][s] = *reinterpret_cast<const h8*>(
              &xs[part * MR * 128 + row * 128 + (((2 * g + s) ^ sx) << 4)]);
        }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int row = 16 * j + r;
      const u4 wq = *reinterpret_cast<const u4*>(&ws[row * 64 + ((g ^ ((row >> 2) & 3)) << 4)]);
      h8 w0, w1;
      widen16(wq, p.flip, c[j], w0, w1);
#pragma unroll
      for (int part = 0; part < (F32 ? 2 : 1); ++part)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          f4v& sum = kLowSums && part ? acc_lo[kLowSums ? i : 0][j] : acc[i][j];
          sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[part][i][0], w0, sum, 0, 0, 0);
          sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[part][i][1], w1, sum, 0, 0, 0);
        }
    }
  };
  // units wave, wave + NW, ... of 64 of k; set u holds unit i + u on its way from memory
  // (past K: zeros, no memory touched).  The scheduling barriers keep a later step's arithmetic
  // on loaded registers from being moved up to where it would wait for their loads.
  const int w64 = __builtin_amdgcn_readfirstlane(wave) * 64;
#pragma unroll
  for (int d = 0; d < D; ++d) fetch(xr[d], wr[d], w64 + d * NW * 64);
  __builtin_amdgcn_sched_barrier(0);
  for (int k0 = w64; k0 < p.K; k0 += D * NW * 64) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      if (u > 0 && k0 + u * NW * 64 >= p.K) break;         // (uniform)
      park(xr[u], wr[u], k0 + u * NW * 64);
      fetch(xr[u], wr[u], k0 + (D + u) * NW * 64);
      multiply();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (kLowSums) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] += acc_lo[i][j];
  }
  // partial sums of the waves through LDS (all waves are done with their pieces of it), a
  // fragment to each of the first MT x FN waves
  __syncthreads();
  float* const red = reinterpret_cast<float*>(wo_lds);   // [MT * FN][NW][4][64]
#pragma unroll
  for (int f = 0; f < MT * FN; ++f)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[((f * NW + wave) * 4 + v) * 64 + lane] = acc[f / FN][f % FN][v];
  __syncthreads();
  if (wave >= MT * FN) return;
  f4v part[NW];
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int v = 0; v < 4; ++v) part[w][v] = red[((wave * NW + w) * 4 + v) * 64 + lane];
  f4v sum = part[0];
  if constexpr (kLowSums) {
    static_assert(NW == 8, "three levels of pairs");
    sum = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
  } else {
#pragma unroll
    for (int w = 1; w < NW; ++w) sum += part[w];
  }
  // D of the 16x16 MFMA: column n = lane % 16, rows 4 (lane / 16) + v
  const int n = n0 + 16 * (wave % FN) + r, m0 = 16 * (wave / FN) + 4 * g;
  if (n >= p.N) return;
  const float sc = to_f32(static_cast<const XT*>(p.scale)[n]);
  const float bi = p.bias ? to_f32(static_cast<const XT*>(p.bias)[n]) : 0.0f;
  XT* out = static_cast<XT*>(p.out);
#pragma unroll
  for (int v = 0; v < 4; ++v)
    if (m0 + v < p.M) out[(int64_t)(m0 + v) * p.ldo + n] = (XT)(sum[v] * sc + bi);
}

// ---------------------------------------------------------------- f32, rows of any length
// f32 activations on rows off 16 bytes, in f32 throughout (v_mfma_f32_32x32x2_f32): 32 rows x 32
// channels per workgroup, k in units of 32 dealt over the waves, operands straight into registers
// -- the 16 MFMAs of a unit take 1024 clocks, its five loads and sixteen conversions a third of
// that.  (One output per thread before: M = 16, 3001 -> 4096 567 us, M = 512, 2047 -> 3001 11.9 ms.)
template <int NW>
__global__ void __launch_bounds__(NW * 64) wo_exact_f32_kernel(const WoParams p) {
  __shared__ float red[NW - 1][16][64];
  typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, g = lane >> 5;
  const int tiles_m = (p.M + 31) / 32;
  const int m0 = (int)(blockIdx.x % tiles_m) * 32, n0 = (int)(blockIdx.x / tiles_m) * 32;
  const int n = min(n0 + r, p.N - 1);
  const float* xrow = static_cast<const float*>(p.x) + (int64_t)min(m0 + r, p.M - 1) * p.ldx;
  const uint8_t* wrow = p.w + (int64_t)n * p.w_sn;
  const int zp = (p.zp ? p.zp[n] : 0) + (p.flip ? 128 : 0);
  f16v acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  f4 xq[2][4];
  u4 wq[2];
  auto fetch = [&](int set, int k0) {                      // lane group g: 16 of the unit's k
    const int k = min(k0 + 16 * g, p.K - 16);
    wq[set] = load_any(wrow, (unsigned)k);
#pragma unroll
    for (int i = 0; i < 4; ++i) xq[set][i] = *reinterpret_cast<const f4_any*>(xrow + k + 4 * i);
  };
  auto multiply = [&](int set, int k0) {
    if (k0 + 32 > p.K) {                                   // (uniform) the end of the rows
      const int z = k0 + 16 * g - min(k0 + 16 * g, p.K - 16);
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (e < z) xq[set][e >> 2][e & 3] = 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int b = (int)(((wq[set][e >> 2] ^ p.flip) >> (8 * (e & 3))) & 0xffu);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xq[set][e >> 2][e & 3], (float)(b - zp), acc, 0, 0, 0);
    }
  };
  const int w32 = __builtin_amdgcn_readfirstlane(wave) * 32;
  fetch(0, w32);
  for (int k0 = w32; k0 < p.K; k0 += 2 * NW * 32) {
    fetch(1, k0 + NW * 32);
    multiply(0, k0);
    fetch(0, k0 + 2 * NW * 32);
    if (k0 + NW * 32 < p.K) multiply(1, k0 + NW * 32);
  }
  if (wave > 0) {
#pragma unroll
    for (int v = 0; v < 16; ++v) red[wave - 1][v][lane] = acc[v];
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int w = 1; w < NW; ++w)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[v] += red[w - 1][v][lane];
    store_frag<float>(p, acc, m0, n0 + r, lane);
  }
}

// ---------------------------------------------------------------- any layout, any alignment
template <typename XT>
__global__ void __launch_bounds__(256) wo_generic_kernel(const WoParams p) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)p.M * p.N) return;
  const int m = (int)(idx / p.N), n = (int)(idx % p.N);
  const XT* x = static_cast<const XT*>(p.x) + (int64_t)m * p.ldx;
  const uint8_t* w = p.w + (int64_t)n * p.w_sn;
  const int zp = p.zp ? p.zp[n] : 0;
  float acc = 0.0f;
  for (int k = 0; k < p.K; ++k) {
    const uint8_t b = w[(int64_t)k * p.w_sk];
    const int q = p.flip ? (int)(int8_t)b : (int)b;
    acc += to_f32(x[k]) * (float)(q - zp);
  }
  const float s = to_f32(static_cast<const XT*>(p.scale)[n]);
  const float b = p.bias ? to_f32(static_cast<const XT*>(p.bias)[n]) : 0.0f;
  static_cast<XT*>(p.out)[(int64_t)m * p.ldo + n] = (XT)(acc * s + b);
}

template <int WM, int FN>
int launch_ragged(dim3 grid, const WoParams& p, hipStream_t st) {
  constexpr int lds = 2 * (WM * 32 + 2 * FN * 32) * 128;
  static_assert(lds <= 64 * 1024, "the stages fit the LDS a launch has without asking");
  hipLaunchKernelGGL((wo_ragged_kernel<WM, FN>), grid, dim3(WM * 128), lds, st, p);
  return check_hip(hipGetLastError(), "dq8_weight_only_qgemm launch");
}

template <typename XT, bool SIGNED, int FM, int NCG, int KG, int BK, int NST, bool WORDS = false>
int launch_dma_kind(const WoParams& p, int splits, hipStream_t st) {
  using Shape = DmaShape<XT, FM, NCG, KG, BK, NST>;
  auto kern = wo_dma_kernel<XT, SIGNED, FM, NCG, KG, BK, NST, WORDS>;
  static std::atomic<uint64_t> lds_allowed{0};
  if (int s = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Shape::kLds, &lds_allowed)) return s;
  const int64_t tiles = ceil_div(p.M, Shape::kBM) * ceil_div(p.N, Shape::kBN);
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)splits), dim3(Shape::kWaves * 64), Shape::kLds, st, p);
  return check_hip(hipGetLastError(), "dq8_weight_only_qgemm launch");
}

template <typename XT, int FM, int NCG, int KG, int BK, int NST>
int launch_dma(const WoParams& p, int splits, hipStream_t st) {
  if constexpr (sizeof(XT) == 2) {
    if (p.words)
      return p.flip ? launch_dma_kind<XT, true, FM, NCG, KG, BK, NST, true>(p, splits, st)
                    : launch_dma_kind<XT, false, FM, NCG, KG, BK, NST, true>(p, splits, st);
  }
  return p.flip ? launch_dma_kind<XT, true, FM, NCG, KG, BK, NST>(p, splits, st)
                : launch_dma_kind<XT, false, FM, NCG, KG, BK, NST>(p, splits, st);
}

template <typename XT, int MR, int U>
int launch_gemv(const WoParams& p, hipStream_t st) {
  const int lds = MR * ((p.K + 7) & ~7) * (int)sizeof(XT);
  auto kern = wo_gemv_kernel<XT, 8, MR, U>;
  static std::atomic<uint64_t> lds_allowed{0};
  if (int s = allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, &lds_allowed)) return s;
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(p.N, 8)), dim3(512), lds, st, p);
  return check_hip(hipGetLastError(), "dq8_weight_only_qgemm launch");
}

template <typename XT, int MT, int FN, bool RAGGED>
int launch_rows_fn(const WoParams& p, hipStream_t st) {
  constexpr int D = sizeof(XT) == 2 && MT == 1 && FN == 1 ? 4 : 2;
  constexpr int lds = kRowsWaves * (MT * 2048 * (int)(sizeof(XT) / 2) + FN * 1024);
  static_assert(lds <= 160 * 1024, "the units fit the LDS");
  auto kern = wo_rows_kernel<XT, MT, FN, D, RAGGED>;
  static std::atomic<uint64_t> lds_allowed{0};
  if (lds > 64 * 1024)
    if (int s = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds, &lds_allowed)) return s;
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(p.N, 16 * FN)), dim3(kRowsWaves * 64), lds, st, p);
  return check_hip(hipGetLastError(), "dq8_weight_only_qgemm launch");
}

template <typename XT, int MT, bool RAGGED>
int launch_rows_mt(const WoParams& p, hipStream_t st) {
  // The workgroup's width: the fewest rounds of the chip, a round priced at the bytes a workgroup
  // stages per unit (weights 16 x 64 a fragment, activations 16 MT x 64 elements).  4096 -> 11008,
  // M = 16, weights from HBM: 16.5 / 16.5 / 13.9 / 15.4 us at 16 / 32 / 48 / 64 channels (three
  // rounds, two, one, one); 4096^2 8.0 / 9.4 / 11.6 / 13.7; 6144^2 16.0 / 13.4 / 16.8 / 19.9.
  const int64_t cus = compute_units(), tiles = ceil_div(p.N, 16);
  int fn = 1;
  int64_t least = INT64_MAX;
  for (int f = 1; f <= 4; ++f) {
    const int64_t t = ceil_div(ceil_div(tiles, f), cus) * (f + MT * (int)sizeof(XT));
    if (t < least) least = t, fn = f;
  }
  // (two 16-channel workgroups share a compute unit: two whole rounds of them are one, and keep more
  // in flight where the rows are deep: 8192^2, M = 16: 20.6 against 21.1 us from HBM, 16.7 against 20.5
  // from the last-level cache; 4096 -> 8192 12.0 / 10.8)
  if (MT == 1 && sizeof(XT) == 2 && p.K >= 8192 && 4 * tiles > 7 * cus && tiles <= 2 * cus) fn = 1;
  switch (fn) {
    case 1: return launch_rows_fn<XT, MT, 1, RAGGED>(p, st);
    case 2: return launch_rows_fn<XT, MT, 2, RAGGED>(p, st);
    case 3: return launch_rows_fn<XT, MT, 3, RAGGED>(p, st);
    default: return launch_rows_fn<XT, MT, 4, RAGGED>(p, st);
  }
}

template <typename XT, bool RAGGED = false>
int launch_rows(const WoParams& p, hipStream_t st) {
  return p.M <= 16 ? launch_rows_mt<XT, 1, RAGGED>(p, st) : launch_rows_mt<XT, 2, RAGGED>(p, st);
}

// The tile forms.  Aligned rows, f16 rows on four bytes: wo_dma_kernel's; f16 rows at other bytes: wo_ragged_kernel's.
enum { kF16_32x64, kF16_64x64, kF16_64x128, kF16_128x128, kF16_128x128Wide, kF16_128x256,
       kF32_32x64, kF32_32x128, kF32_64x128, kF32_64x128Wide, kF32_64x256,
       kRagged64x64, kRagged128x128, kNumForms };

// Estimated time of a plan in microseconds,
//   t = c0 + kt (c1 + c2 (r - 1)) + c3 (r - 1) + [splits > 1] (c4 + c5 M N splits / 1e6) + c6 M N / 1e6
// kt: 64-deep k tiles per workgroup; r: workgroups per compute unit, rounded up.  Fitted (least
// squares on relative error, median error 4 %, 90th percentile 11 %) to 32800 timed launches of the
// f16 forms and 24000 of the f32 forms: M = 33 .. 2048, K = 512 .. 8192, N = 512 .. 11008, odd sizes
// among them, 1 .. 8 k ranges; the ragged forms to 3300 of their aligned forerunners.
struct TileForm { int bm, bn; float c0, c1, c2, c3, c4, c5, c6; };
constexpr TileForm kForms[kNumForms] = {
    {32, 64, 4.034f, 0.119f, 0.104f, 0.002f, 2.743f, 1.841f, 1.814f},
    {64, 64, 4.606f, 0.160f, 0.148f, -0.117f, 2.828f, 2.293f, 1.506f},
    {64, 128, 5.183f, 0.249f, 0.239f, -0.407f, 2.746f, 2.327f, 1.052f},
    {128, 128, 5.955f, 0.324f, 0.362f, -1.529f, 2.921f, 2.188f, 1.186f},
    {128, 128, 6.834f, 0.291f, 0.428f, 0.751f, 2.880f, 2.369f, 1.249f},
    {128, 256, 7.976f, 0.505f, 0.831f, -2.607f, 3.172f, 1.979f, 1.068f},
    {32, 64, 4.606f, 0.175f, 0.185f, 1.795f, 2.426f, 2.974f, 2.336f},
    {32, 128, 4.854f, 0.236f, 0.298f, 1.117f, 2.514f, 3.206f, 2.262f},
    {64, 128, 5.656f, 0.402f, 0.407f, -1.281f, 2.713f, 2.353f, 1.852f},
    {64, 128, 5.810f, 0.345f, 0.482f, 0.446f, 2.714f, 2.864f, 2.221f},
    {64, 256, 6.141f, 0.614f, 0.895f, -2.083f, 2.916f, 2.498f, 2.051f},
    {64, 64, 4.272f, 0.274f, 0.177f, 0.472f, 2.347f, 1.649f, 0.0f},
    {128, 128, 7.616f, 0.569f, 0.484f, -0.948f, 1.629f, 1.696f, 0.0f},
};

// Plan: `splits` workgroups per tile of form `form`, each over k_split of the k range, and
// (splits > 1) a reduction kernel behind them.  `us`: the estimate it was chosen by.
struct SplitPlan {
  int form;
  int splits;
  int k_split;
  float us;
};

// The cheapest of the type's forms with 1, 2, 3, 4, 6 or 8 k ranges of at least 192, from `least`
// ranges on and up to `most`.  Choosing by this estimate comes within 0.8 % (geometric mean; 95 %
// within 5 %) of the best timed plan of each of the 3400 problems it was fitted to.
SplitPlan plan_split(int64_t M, int64_t N, int64_t K, int esz, bool ragged, int least, int most) {
  SplitPlan best = {-1, 1, (int)K, 0.0f};
  const int64_t cus = compute_units();
  const int first = ragged ? kRagged64x64 : esz == 4 ? kF32_32x64 : kF16_32x64;
  const int last = ragged ? kRagged128x128 : esz == 4 ? kF32_64x256 : kF16_128x256;
  for (int form = first; form <= last; ++form) {
    const TileForm& c = kForms[form];
    const int64_t tiles = ceil_div(M, c.bm) * ceil_div(N, c.bn);
    const float mn = (float)((double)M * (double)N * 1e-6);
    for (int want : {1, 2, 3, 4, 6, 8}) {
      if (want > most || (want > 1 && K / want < 192)) break;
      const int64_t k_split = ceil_div(ceil_div(K, (int64_t)want), 64) * 64;
      const int64_t splits = ceil_div(K, k_split);
      if (splits < least) continue;
      const float kt = (float)(k_split / 64), r = (float)(ceil_div(tiles * splits, cus) - 1);
      float us = c.c0 + kt * (c.c1 + c.c2 * r) + c.c3 * r + c.c6 * mn;
      if (splits > 1) us += c.c4 + c.c5 * mn * (float)splits;
      if (best.form < 0 || us < best.us)
        best = {form, (int)splits, splits > 1 ? (int)k_split : (int)K, us};
    }
  }
  return best;
}

// Whether 17 .. 32 rows of f32 run on tiles.  us at 24 rows, staged / tiles: 4104 channels (from 4097 on the
// staged kernel's workgroups are 32 wide) 256 of k 4.70 / 4.15, 448 5.0 / 5.05, 768 5.7 / 6.45, 1024 6.1 / 7.1,
// 2048 8.7 / 9.9; 8192 channels 256 4.8 / 4.25, 512 5.3 / 5.4, 1024 6.7 / 7.3, 2304 9.7 / 10.8, 2816 equal, 4096
// 16.3 / 14.4; 9216 and more equal at 768 to 2048, tiles 1.06-1.24 times as fast on either side.  Up to 4096
// channels tiles win from 3584 of k on (4096^2 13.1 / 12.0); from 2048 on, and to 6143 channels, they are
// taken for their sums: split over k, 0.97e-7 rms against 64 bits where the staged kernel has 1.6e-7 (one
// sum for both halves) and 1.03e-7, for 0.05-0.2 of the time.
bool f32_rows_on_tiles(int64_t N, int64_t K) {
  if (N > 8192 || (N > 4096 && K < 400)) return true;
  return K > (N >= 6144 ? 2816 : 2048);
}

// The plan for M x N x K, or form = -1 where the kernels for few rows are the choice: up to 32 rows, for
// f32 up to 16 where the staged kernel, which multiplies two half tiles, is the slower or less exact one
// (f16 up to 32 rows, tiles against the staged kernel: 0.65-0.95 times as fast).
SplitPlan choose_tiles(int64_t M, int64_t N, int64_t K, int esz, bool ragged, int most_splits) {
  const SplitPlan none = {-1, 1, (int)K, 0.0f};
  // (rows off 16 bytes: f16 has tiles and the staged small-M kernel, f32 its own kernel)
  if (ragged && (esz == 4 || M <= 32)) return none;
  if (M <= (esz == 4 && f32_rows_on_tiles(N, K) ? 16 : 32)) return none;
  return plan_split(M, N, K, esz, ragged, 1, most_splits);
}

size_t split_bytes(const SplitPlan& s, int64_t M, int64_t N) {
  return s.splits > 1 ? (size_t)s.splits * (size_t)(M * N) * sizeof(float) : 0;
}

// The operands' rows are not multiples of 16 bytes, 16-byte aligned.
bool rows_ragged(const void* x, int esz, int64_t ldx, const void* w, int64_t w_sn, int64_t K) {
  return !(K % 16 == 0 && aligned(x, 16) && (ldx * esz) % 16 == 0 && aligned(w, 16) && w_sn % 16 == 0);
}

// (the tiles address their rows by 31-bit byte offsets from the first)
bool tiles_reach(int64_t ldx, int64_t w_sn, int64_t K) {
  return 512 * ldx + 4 * K + 4096 < (1LL << 31) && 256 * w_sn + K + 4096 < (1LL << 31);
}

// one launch of a form over the whole k range (splits == 1) or its split
template <typename XT>
int launch_form(int form, int splits, const WoParams& p, hipStream_t st) {
  if constexpr (sizeof(XT) == 2) {
    const dim3 grid((unsigned)(ceil_div(p.M, kForms[form].bm) * ceil_div(p.N, kForms[form].bn)), (unsigned)splits);
    switch (form) {
      case kF16_32x64: return launch_dma<XT, 1, 1, 4, 128, 4>(p, splits, st);
      case kF16_64x64: return launch_dma<XT, 2, 1, 4, 128, 3>(p, splits, st);
      case kF16_64x128: return launch_dma<XT, 2, 2, 2, 64, 4>(p, splits, st);
      case kF16_128x128: return launch_dma<XT, 4, 2, 2, 64, 3>(p, splits, st);
      case kF16_128x128Wide: return launch_dma<XT, 4, 2, 4, 128, 3>(p, splits, st);
      case kF16_128x256: return launch_dma<XT, 4, 4, 2, 64, 4>(p, splits, st);
      case kRagged64x64: return launch_ragged<2, 1>(grid, p, st);
      case kRagged128x128: return launch_ragged<4, 2>(grid, p, st);
    }
  } else {
    switch (form) {
      case kF32_32x64: return launch_dma<XT, 1, 1, 4, 128, 4>(p, splits, st);
      case kF32_32x128: return launch_dma<XT, 1, 2, 4, 128, 4>(p, splits, st);
      case kF32_64x128: return launch_dma<XT, 2, 2, 2, 64, 3>(p, splits, st);
      case kF32_64x128Wide: return launch_dma<XT, 2, 2, 4, 128, 3>(p, splits, st);
      case kF32_64x256: return launch_dma<XT, 2, 4, 2, 64, 4>(p, splits, st);
    }
  }
  return fail("dq8_weight_only_qgemm: unknown tile form");
}

template <typename XT>
int launch(WoParams& p, bool fast, void* scratch, size_t scratch_bytes, hipStream_t st) {
  p.partial = nullptr;
  p.k_split = p.K;
  if (fast && tiles_reach(p.ldx, p.w_sn, p.K)) {
    const bool have = scratch && aligned(scratch, 16);
    const size_t planes = have ? scratch_bytes / ((size_t)p.M * (size_t)p.N * sizeof(float)) : 0;
    // (unaligned rows whose scratch was sized for aligned ones: as many k ranges as it holds)
    // (rows on four bytes: the aligned rows' tiles, in the scratch that the ragged ones ask for: 2052 of k, 128 x 4096
    // 13.1 -> 8.5 us, 700 x 4096 30.5 -> 22.3, 300 x 1000 11.1 -> 8.3)
    const bool ragged = p.ragged && !p.words;
    SplitPlan s = choose_tiles(p.M, p.N, p.K, (int)sizeof(XT), ragged,
                               p.ragged ? (int)std::min<size_t>(std::max<size_t>(planes, 1), 8) : have ? 8 : 1);
    if (s.splits > 1 && scratch_bytes < split_bytes(s, p.M, p.N))
      s = choose_tiles(p.M, p.N, p.K, (int)sizeof(XT), ragged, 1);
    if (s.form >= 0 && s.splits > 1) {
      const int sp = s.splits;
      p.partial = static_cast<float*>(scratch);
      p.k_split = s.k_split;
      if (int e = launch_form<XT>(s.form, sp, p, st)) return e;
      const int vec = (p.N % 4 == 0 && aligned(p.out, 8) && p.ldo % 4 == 0) ? 4 : 1;
      const int64_t blocks = ceil_div((int64_t)p.M * (p.N / vec), 256);
      DQ8_REQUIRE(blocks < (1LL << 31), "dq8_weight_only_qgemm: problem too large");
      if (vec == 4)
        hipLaunchKernelGGL((wo_splitk_reduce_kernel<XT, 4>), dim3((unsigned)blocks), dim3(256), 0,
                           st, p, sp);
      else
        hipLaunchKernelGGL((wo_splitk_reduce_kernel<XT, 1>), dim3((unsigned)blocks), dim3(256), 0,
                           st, p, sp);
      return check_hip(hipGetLastError(), "dq8_weight_only_qgemm reduction launch");
    }
    if (s.form >= 0) return launch_form<XT>(s.form, 1, p, st);
  }
  // (the staged kernel addresses activation and weight rows by 31-bit byte offsets)
  const bool staged_ok =
      ((int64_t)(p.M - 1) * p.ldx + p.K) * (int64_t)sizeof(XT) + 65536 < (1LL << 31) &&
      64 * p.w_sn + (int64_t)p.K + 65536 < (1LL << 31);
  if (fast && p.ragged) {
    if constexpr (sizeof(XT) == 4) {
      const int64_t tiles = ceil_div(p.M, 32) * ceil_div(p.N, 32);
      // (few tiles: eight waves share the k range, so that most compute units' matrix cores run)
      if (tiles <= 4 * compute_units()) {
        hipLaunchKernelGGL(wo_exact_f32_kernel<8>, dim3((unsigned)tiles), dim3(512), 0, st, p);
        return check_hip(hipGetLastError(), "dq8_weight_only_qgemm launch");
      }
      if (tiles < (1LL << 31)) {
        hipLaunchKernelGGL(wo_exact_f32_kernel<4>, dim3((unsigned)tiles), dim3(256), 0, st, p);
        return check_hip(hipGetLastError(), "dq8_weight_only_qgemm launch");
      }
    } else if (staged_ok && p.M <= 32) {
      return launch_rows<XT, true>(p, st);
    }
    fast = false;
  }
  if (!fast) {
    const int64_t blocks = ceil_div((int64_t)p.M * p.N, 256);
    DQ8_REQUIRE(blocks < (1LL << 31), "dq8_weight_only_qgemm: problem too large");
    hipLaunchKernelGGL(wo_generic_kernel<XT>, dim3((unsigned)blocks), dim3(256), 0, st, p);
  } else if (p.M <= 128) {
    // One row, and two where it was measured faster, while the rows fit 64 KiB of LDS: the
    // row-streaming kernel on the vector ALUs (4096^2 weights, M = 1: f16 4.3 us, f32 4.5; M = 2, weights
    // from HBM, against the kernel below: 3072 -> 768 f16 5.1 / 5.3 us, f32 5.3 / 6.5; 8192 -> 1024 f32
    // 8.8 / 12.0; 4096^2 f16 7.9 / 7.4, f32 8.5 / 8.7; 4096 -> 11008 f16 14.2 / 13.2, f32 15.3 / 14.1;
    // 8192^2 from the last-level cache f32 20.0 / 20.9).
    const bool two = sizeof(XT) == 4 ? p.N < 8192 || p.K > 4096 : p.N <= 1024 && p.K >= 2048 && p.K <= 8192;
    if ((p.M == 1 || (p.M == 2 && two)) && (int64_t)p.M * p.K * (int64_t)sizeof(XT) <= 64 * 1024) {
      const bool deep = p.K > 4096;
      if (p.M == 1) return deep ? launch_gemv<XT, 1, 8>(p, st) : launch_gemv<XT, 1, 4>(p, st);
      return deep ? launch_gemv<XT, 2, 8>(p, st) : launch_gemv<XT, 2, 4>(p, st);
    }
    // Up to 32 rows: the staged kernel (against kernels that gathered both operands lane by lane, weights
    // from HBM, f16: 1024 -> 11008 M = 16 9.3 -> 6.3 us, 1536 -> 6144 M = 8 6.5 -> 5.8, M = 32 9.0 ->
    // 7.2, 3072 -> 768 M = 4 6.4 -> 5.5; f32: 768 -> 3072 M = 16 5.7 -> 4.9, M = 32 8.9 -> 6.7).
    if (staged_ok && p.M <= 32) return launch_rows<XT>(p, st);
    const unsigned grid = (unsigned)ceil_div(p.N, 32);
    if (p.M <= 32)
      hipLaunchKernelGGL((wo_skinny_kernel<XT, 8, 1>), dim3(grid), dim3(512), 0, st, p);
    else if (p.M <= 64)
      hipLaunchKernelGGL((wo_skinny_kernel<XT, 8, 2>), dim3(grid), dim3(512), 0, st, p);
    else
      hipLaunchKernelGGL((wo_skinny_kernel<XT, 8, 4>), dim3(grid), dim3(512), 0, st, p);
  } else {
    // (the LDS kernels cannot address the operands: the register kernel)
    const int64_t big = ceil_div(p.M, 128) * ceil_div(p.N, 128);
    if (big >= 192) {
      hipLaunchKernelGGL((wo_tile_kernel<XT, 2, 2>), dim3((unsigned)big), dim3(256), 0, st, p);
    } else {
      const int64_t small = ceil_div(p.M, 64) * ceil_div(p.N, 64);
      hipLaunchKernelGGL((wo_tile_kernel<XT, 1, 1>), dim3((unsigned)small), dim3(256), 0, st, p);
    }
  }
  return check_hip(hipGetLastError(), "dq8_weight_only_qgemm launch");
}

}  // namespace

void weight_only_plan(int64_t M, int64_t N, int64_t K, int esz, bool ragged, int plan[4]) {
  const SplitPlan s = choose_tiles(M, N, K, esz, ragged, 8);
  plan[0] = s.form;
  plan[1] = s.splits;
  plan[2] = s.form < 0 ? 0 : kForms[s.form].bm;
  plan[3] = s.form < 0 ? 0 : kForms[s.form].bn;
}

}  // namespace dq8

using namespace dq8;

namespace {
// bytes of the [N, K] copy of weights given as [K, N], kept 256-byte aligned
size_t transposed_bytes(int64_t N, int64_t K, int tp_b) {
  return (tp_b || N <= 0 || K <= 0) ? 0 : ((size_t)(N * K) + 255) / 256 * 256;
}
// Undoes the byte permutation the reference's compiler applies to a constant [K, N] ui8 weight
// (R tao_compiler/mlir/disc/transforms/disc_transform_weight_data_layout_for_weight_only_gemm.cc
// :54-300 as composed at :362-370: rows permuted in blocks of 16, transpose, column pairs
// interleaved in tiles of 64 rows, bytes 1 and 2 of every word swapped).  Composed, the 16
// bytes W^T[n, 16 j .. 16 j + 15] sit in one 16-byte group of the reordered buffer, at byte
//   (n / 2) * 2 K + (16 j / 64) * 128 + (n % 2) * 64 + (16 j) % 64,
// even bytes of the group = the first eight k, odd bytes = the last eight.  One thread per
// group: a 16-byte load, four byte permutes, a 16-byte store into the kernels' [N, K] layout.
__global__ void __launch_bounds__(256)
wo_undo_compiler_layout_kernel(const u4* __restrict__ src, u4* __restrict__ dst, int N, int K16) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (g >= (int64_t)N * K16) return;
  const int n = (int)(g / K16), j = (int)(g % K16);
  const int64_t off16 = (int64_t)(n >> 1) * (2 * K16) + (j >> 2) * 8 + (n & 1) * 4 + (j & 3);
  const u4 v = __builtin_nontemporal_load(src + off16);
  u4 r;
  // v_perm_b32 selector bytes: 0-3 pick from the second operand, 4-7 from the first
  r.x = __builtin_amdgcn_perm(v.y, v.x, 0x06040200u);   // k 0..3  = bytes 0,2 of words 0,1
  r.y = __builtin_amdgcn_perm(v.w, v.z, 0x06040200u);   // k 4..7  = bytes 0,2 of words 2,3
  r.z = __builtin_amdgcn_perm(v.y, v.x, 0x07050301u);   // k 8..11 = bytes 1,3 of words 0,1
  r.w = __builtin_amdgcn_perm(v.w, v.z, 0x07050301u);   // k 12..15
  dst[g] = r;
}

}  // namespace

extern "C" size_t dq8_weight_only_qgemm_workspace_bytes(int64_t N, int64_t K, int tp_b) {
  return (tp_b || N <= 0 || K <= 0) ? 0 : (size_t)(N * K);
}

namespace {
// The [N, K] copy of weights given as [K, N], and the partial sums of the plan that the call then takes.
size_t scratch_bytes(int64_t M, int64_t N, int64_t K, int tp_b, int x_dtype, bool ragged) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  size_t split = 0;
  if ((x_dtype == DQ8_DTYPE_F16 || x_dtype == DQ8_DTYPE_F32) && K >= 16 && M < (1LL << 31) &&
      N < (1LL << 31) && K < (1LL << 31))
    split = split_bytes(choose_tiles(M, N, K, x_dtype == DQ8_DTYPE_F32 ? 4 : 2, ragged, 8), M, N);
  if (!split) return dq8_weight_only_qgemm_workspace_bytes(N, K, tp_b);
  return transposed_bytes(N, K, tp_b) + split;
}
}  // namespace

extern "C" size_t dq8_weight_only_qgemm_workspace_bytes_ex(int64_t M, int64_t N, int64_t K,
                                                           int tp_b, int x_dtype) {
  return scratch_bytes(M, N, K, tp_b, x_dtype, K % 16 != 0);
}

extern "C" size_t dq8_weight_only_qgemm_workspace_bytes_for(const void* x, int x_dtype, int64_t ldx, const void* w,
                                                            int64_t ldw, int tp_b, int64_t M, int64_t N, int64_t K) {
  const int64_t w_sn = tp_b ? ldw : K;                     // (the copy's rows follow each other)
  if (!tiles_reach(ldx, w_sn, K)) return dq8_weight_only_qgemm_workspace_bytes(N, K, tp_b);
  return scratch_bytes(M, N, K, tp_b, x_dtype,
                       rows_ragged(x, x_dtype == DQ8_DTYPE_F32 ? 4 : 2, ldx, tp_b ? w : nullptr, w_sn, K));
}

extern "C" int dq8_weight_only_undo_compiler_layout(const uint8_t* reordered, uint8_t* w_nk,
                                                    int64_t K, int64_t N, void* stream) {
  clear_error();
  DQ8_REQUIRE(K >= 0 && N >= 0 && K < (1LL << 31) && N < (1LL << 31),
              "dq8_weight_only_undo_compiler_layout: bad shape");
  // (outside these shapes the compiler's pass reads and writes out of bounds: not a permutation)
  DQ8_REQUIRE(K % 64 == 0 && N % 4 == 0,
              "dq8_weight_only_undo_compiler_layout: the compiler's weight layout is defined for "
              "K % 64 == 0 and N % 4 == 0 only");
  if (K == 0 || N == 0) return 0;
  DQ8_REQUIRE(reordered && w_nk, "dq8_weight_only_undo_compiler_layout: null pointer");
  DQ8_REQUIRE(aligned(reordered, 16) && aligned(w_nk, 16),
              "dq8_weight_only_undo_compiler_layout: buffers must be 16-byte aligned");
  DQ8_REQUIRE(reordered != w_nk, "dq8_weight_only_undo_compiler_layout: not in place");
  const int64_t groups = N * (K / 16);
  hipLaunchKernelGGL(wo_undo_compiler_layout_kernel, dim3((unsigned)ceil_div(groups, 256)),
                     dim3(256), 0, (hipStream_t)stream, reinterpret_cast<const u4*>(reordered),
                     reinterpret_cast<u4*>(w_nk), (int)N, (int)(K / 16));
  return check_hip(hipGetLastError(), "dq8_weight_only_undo_compiler_layout launch");
}

extern "C" int dq8_weight_only_qgemm(const void* x, int x_dtype, int64_t ldx, const void* w,
                                     int w_signed, int64_t ldw, int tp_b, const void* scale,
                                     const int32_t* zero_points, const void* bias, void* out,
                                     int64_t ldo, int64_t M, int64_t N, int64_t K,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  DQ8_REQUIRE(x_dtype == DQ8_DTYPE_F32 || x_dtype == DQ8_DTYPE_F16,
              "dq8_weight_only_qgemm: activations must be f32 or f16");
  DQ8_REQUIRE(M >= 0 && N >= 0 && K >= 0, "dq8_weight_only_qgemm: negative size");
  DQ8_REQUIRE(M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31),
              "dq8_weight_only_qgemm: size too large");
  if (M == 0 || N == 0) return 0;
  DQ8_REQUIRE(x && w && scale && out, "dq8_weight_only_qgemm: null pointer");
  DQ8_REQUIRE(ldx >= K && ldo >= N && ldw >= (tp_b ? K : N),
              "dq8_weight_only_qgemm: leading dimension too small");
  hipStream_t st = (hipStream_t)stream;
  const int esz = x_dtype == DQ8_DTYPE_F32 ? 4 : 2;
  WoParams p;
  p.x = x;
  p.w = static_cast<const uint8_t*>(w);
  p.scale = scale;
  p.zp = zero_points;
  p.bias = bias;
  p.out = out;
  p.ldx = ldx;
  p.ldo = ldo;
  p.w_sn = tp_b ? ldw : 1;
  p.w_sk = tp_b ? 1 : ldw;
  p.M = (int)M;
  p.N = (int)N;
  p.K = (int)K;
  p.flip = w_signed ? 0x80808080u : 0u;
  // the MFMA kernels want k-contiguous rows of both operands, of at least 16 elements; weights given
  // as [K, N] are transposed into the caller's scratch first (a runtime does that once per
  // constant weight and passes the result with tp_b = 1 from then on)
  bool fast = K >= 16;
  // what the transposed weights leave of the scratch holds the partial sums of a split launch
  void* rest = workspace;
  size_t rest_bytes = workspace ? workspace_bytes : 0;
  if (fast && !tp_b) {
    if (workspace && aligned(workspace, 16) && workspace_bytes >= (size_t)(N * K)) {
      if (int s = dq8_transpose_s8(static_cast<const int8_t*>(w), ldw,
                                   static_cast<int8_t*>(workspace), K, N, stream))
        return s;
      p.w = static_cast<const uint8_t*>(workspace);
      p.w_sn = K;
      p.w_sk = 1;
      const size_t used = transposed_bytes(N, K, 0);
      rest = used < workspace_bytes ? static_cast<char*>(workspace) + used : nullptr;
      rest_bytes = used < workspace_bytes ? workspace_bytes - used : 0;
    } else {
      fast = false;
    }
  }
  fast = fast && p.w_sk == 1;
  p.ragged = rows_ragged(x, esz, ldx, p.w, p.w_sn, K);
  p.words = p.ragged && esz == 2 && K >= 64 && K % 4 == 0 && ldx % 2 == 0 && p.w_sn % 4 == 0 && aligned(x, 4) &&
            aligned(p.w, 4);
  return x_dtype == DQ8_DTYPE_F32 ? launch<float>(p, fast, rest, rest_bytes, st)
                                  : launch<_Float16>(p, fast, rest, rest_bytes, st);
}
