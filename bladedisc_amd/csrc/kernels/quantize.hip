// quantize / dequantize for gfx950: bandwidth-bound, 5 bytes of HBM traffic per
// element.  Semantics follow the reference's runtime decomposition of
// mhlo_disc.quantize / mhlo_disc.dequantize
// (tao_compiler/mlir/disc/transforms/disc_lower_quantize_and_dequantize.cc:77-94,
// 131-136): every step is a separately rounded binary32 operation and the
// division is a true IEEE division, so this file is compiled with
// -ffp-contract=off.
//
// Access patterns:
//   per tensor            1-D sweep over float4 / packed-4 elements
//   per channel, inner==1 (channel is the last axis) 2-D tiles [rows, 4*threads];
//                         each thread keeps its four scales / zero points in
//                         registers while it walks down the rows
//   per channel, inner%4==0 one (outer, channel) row per blockIdx.y
// for f32 and the 8-bit types at sizes that are multiples of four; every other type, size and
// alignment runs the general kernels, in groups of four elements as well (lastaxis_any; sweep_any
// along the last axis or per tensor; rows_any on other axes; flat_any for the rest).
#include <algorithm>

#include <cstdlib>
#include "dq8_common.h"
#include "disc_q8.h"
#include "q8_elementwise.h"

#pragma clang fp contract(off)

namespace {

using namespace dq8::elementwise;

// Four values quantized with one divisor (or one per component) through its reciprocal: the
// quotients are the bits of x / s (div4_by_constant), so the result is quant_one's; with
// half-to-even rounding, clamping, rounding and byte packing are the epilogue's v_med3 + SDWA
// add.  About 7 vector instructions per element instead of 19 -- with the true division quantize
// was as close to the VALU's limit as to the memory's.
template <int ROUND>
__device__ __forceinline__ uint32_t finish4_quotients(const float4& t, float lo, float hi) {
  if (ROUND == 1) return quant4_pack_rne(t, lo, hi);
  return pack4(quant_from_quotient<ROUND>(t.x, lo, hi), quant_from_quotient<ROUND>(t.y, lo, hi),
               quant_from_quotient<ROUND>(t.z, lo, hi), quant_from_quotient<ROUND>(t.w, lo, hi));
}
template <int ROUND>
__device__ __forceinline__ uint32_t quant4_by_constant(const float4& v, float s, float y, float z,
                                                       float lo, float hi) {
  const float4 q = div4_by_constant(v, s, y);
  return finish4_quotients<ROUND>(make_float4(q.x + z, q.y + z, q.z + z, q.w + z), lo, hi);
}
template <int ROUND>
__device__ __forceinline__ uint32_t quant4_by_constants(const float4& v, const float4& s,
                                                        const float4& y, const float4& z,
                                                        float lo, float hi) {
  const float4 q = div4_by_constants(v, s, y);
  return finish4_quotients<ROUND>(make_float4(q.x + z.x, q.y + z.y, q.z + z.z, q.w + z.w), lo, hi);
}

// Workgroups go to the eight accelerator dies in turn.  The sweeps take chunks of kThreads groups of four,
// chunk j on die j % 8 whatever the type and however many chunks a thread takes (kHop groups apart): what
// one of them has just written the next one finds in its die's L2, and one chunk to a workgroup is the
// plain linear order.  Quantize and dequantize in one buffer, us, with contiguous chunks / with these, f32
// through int8: 1000 x 3072 11.6 / 8.8, 2000 x 3072 20.6 / 9.7, 5400 x 3072 31.9 / 28.3, 8000 x 3072 41.5 /
// 40.2; f16 through int8 3000 x 3072 17.8 / 11.4.
constexpr int kHop = 8 * kThreads;
template <int U>
__device__ __forceinline__ uint32_t sweep_first_group() {
  const uint32_t b = blockIdx.x;
  return (U == 1 ? b : b / 8 * (8 * U) + b % 8) * kThreads + threadIdx.x;
}
template <int U>
unsigned sweep_workgroups(int64_t n) {           // (one group more: the elements behind the last four)
  const int64_t chunks = dq8::ceil_div(n / 4 + 1, (int64_t)kThreads);
  return (unsigned)(U == 1 ? chunks : dq8::ceil_div(chunks, (int64_t)(8 * U)) * 8);
}
// The 8-bit results of a tensor that the eight L2s, 4 MiB each, can still hold in part when the next
// operator reads them.  (Beyond, dequantize's two chunks next to each other: 16000 x 3072 34.6 us, 35.0 with
// them kHop apart.)
inline bool l2s_hold(int64_t n) { return n <= (1 << 25); }

// ---------------------------------------------------------------- per tensor
// One unit per thread and a grid that covers the tensor in one sweep (the loop only
// runs again beyond 2^30 units): on this part a linear sweep by many small workgroups
// reaches more of the HBM bandwidth than fewer workgroups that each keep several
// far-apart streams in flight (measured on 1 GiB of f32: 6.2 TB/s against 4.7-5.2).
template <int ROUND>
__global__ void __launch_bounds__(kThreads)
quantize_tensor_v4(const float4* __restrict__ x, uint32_t* __restrict__ out,
                   int64_t n, const float* __restrict__ scale,
                   const int32_t* __restrict__ zp, float lo, float hi) {
  const int64_t n4 = n >> 2;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i < n4) {
    // The data load goes out first: a wave has one load to make, and behind the scalar loads of
    // the parameters and the reciprocal it would start a cache miss later.
    float4 v = x[i];
    __builtin_amdgcn_sched_barrier(0);
    const float s = scale[0];
    const float z = (float)zp[0];
    const float y = 1.0f / s;
    const bool fast = divisor_in_fast_range(s);
    for (;;) {
      out[i] = fast ? quant4_by_constant<ROUND>(v, s, y, z, lo, hi)
                    : pack4(quant_one<ROUND>(v.x, s, z, lo, hi), quant_one<ROUND>(v.y, s, z, lo, hi),
                            quant_one<ROUND>(v.z, s, z, lo, hi), quant_one<ROUND>(v.w, s, z, lo, hi));
      i += stride;
      if (i >= n4) break;
      v = x[i];
    }
  }
  if (i - n4 < (n & 3)) {                  // the up to three elements behind the last four
    const int64_t e = i + 3 * n4;
    reinterpret_cast<uint8_t*>(out)[e] = (uint8_t)quant_one<ROUND>(
        reinterpret_cast<const float*>(x)[e], scale[0], (float)zp[0], lo, hi);
  }
}

template <bool SIGNED>
__device__ __forceinline__ float4 dequant_word(uint32_t w, int z, float s) {
  const int4 b = unpack4<SIGNED>(w);
  return make_float4((float)(b.x - z) * s, (float)(b.y - z) * s, (float)(b.z - z) * s,
                     (float)(b.w - z) * s);
}

template <bool SIGNED>
__device__ __forceinline__ float4 dequant_word4(uint32_t w, const int4& z, const float4& s) {
  const int4 b = unpack4<SIGNED>(w);
  return make_float4((float)(b.x - z.x) * s.x, (float)(b.y - z.y) * s.y,
                     (float)(b.z - z.z) * s.z, (float)(b.w - z.w) * s.w);
}

// Two 4-byte words in, two 16-byte stores out per thread, one sweep.  A workgroup covers two chunks of
// 256 consecutive words, HOP words apart (kThreads or kHop), and a thread takes word t of each, so that
// every load and store instruction of a wave covers one contiguous span (64 x 16 bytes per store).  With the
// two words of a thread next to each other (one 8-byte load, stores 32 bytes apart between
// neighbouring lanes) tensors that fit the last-level cache ran a quarter slower:
// [4096,768] 5.35 -> 4.3 us, [32,56,56,64] 8.1 -> 6.1 us, [65536,4096] 221 -> 210 us.
// The f32 results leave with the streaming hint (every store instruction is a whole kilobyte):
// [4096,768] 4.37 -> 3.35 us, [32,56,56,64] 6.3 -> 5.1 us, [65536,4096] 216 -> 187 us, which
// is 7.2 TB/s; the same hint on the loads made every size slower, and on quantize's stores (a
// fifth of its traffic) it helped some sizes and hurt others, so neither is used.
template <bool SIGNED, int HOP>
__global__ void __launch_bounds__(kThreads)
dequantize_tensor_v4x2(const uint32_t* __restrict__ q, float4* __restrict__ out,
                       int64_t n, const float* __restrict__ scale,
                       const int32_t* __restrict__ zp) {
  const float s = scale[0];
  const int z = zp[0];
  const int64_t n4 = n >> 2;
  const int64_t stride = (int64_t)gridDim.x * (2 * kThreads);
  for (int64_t i = HOP == kHop ? (int64_t)sweep_first_group<2>() : (int64_t)blockIdx.x * (2 * kThreads) + threadIdx.x;
       i < n4; i += stride) {
    const bool two = i + HOP < n4;
    const uint32_t w0 = q[i];
    const uint32_t w1 = two ? q[i + HOP] : 0u;
    dq8::st_stream(&out[i], dequant_word<SIGNED>(w0, z, s));
    if (two) dq8::st_stream(&out[i + HOP], dequant_word<SIGNED>(w1, z, s));
  }
  if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {        // the elements behind the last word
    const int64_t e = 4 * n4 + threadIdx.x;
    const uint8_t b = reinterpret_cast<const uint8_t*>(q)[e];
    reinterpret_cast<float*>(out)[e] = (float)((SIGNED ? (int)(int8_t)b : (int)b) - z) * s;
  }
}

// ------------------------------------------- per channel, channel = last axis
// x: [rows, nch], nch % 4 == 0.  threadIdx.x / blockIdx.x tile channels (4 per thread),
// threadIdx.y / blockIdx.y tile rows: each block walks rows_per_block rows, blockDim.y at
// a time (tensors with few channels put several rows side by side in one workgroup).
template <int ROUND>
__global__ void __launch_bounds__(kThreads)
quantize_lastaxis_v4(const float4* __restrict__ x, uint32_t* __restrict__ out,
                     int64_t rows, int nch4, int rows_per_block,
                     const float4* __restrict__ scale,
                     const int4* __restrict__ zp, float lo, float hi) {
  const int c4 = blockIdx.x * blockDim.x + threadIdx.x;
  if (c4 >= nch4) return;
  const float4 s = scale[c4];
  const int4 zi = zp[c4];
  const float4 z = make_float4((float)zi.x, (float)zi.y, (float)zi.z, (float)zi.w);
  const int64_t r_begin = (int64_t)blockIdx.y * rows_per_block;
  const int64_t r_end = r_begin + rows_per_block < rows ? r_begin + rows_per_block : rows;
  const int64_t step = blockDim.y;               // rows between two rows of this thread
  const int64_t hop = step * nch4;               // the same in units
  int64_t r = r_begin + threadIdx.y;
  const float4* px = x + r * nch4 + c4;
  uint32_t* po = out + r * nch4 + c4;
  const float4 y = make_float4(1.0f / s.x, 1.0f / s.y, 1.0f / s.z, 1.0f / s.w);
  const bool fast = divisor_in_fast_range(s.x) && divisor_in_fast_range(s.y) &&
                    divisor_in_fast_range(s.z) && divisor_in_fast_range(s.w);
  auto one = [&](const float4& v) {
    if (fast) return quant4_by_constants<ROUND>(v, s, y, z, lo, hi);
    return pack4(quant_one<ROUND>(v.x, s.x, z.x, lo, hi), quant_one<ROUND>(v.y, s.y, z.y, lo, hi),
                 quant_one<ROUND>(v.z, s.z, z.z, lo, hi), quant_one<ROUND>(v.w, s.w, z.w, lo, hi));
  };
  for (; r + 3 * step < r_end; r += 4 * step, px += 4 * hop, po += 4 * hop) {
    const float4 v0 = px[0], v1 = px[hop], v2 = px[2 * hop], v3 = px[3 * hop];
    dq8::st_stream(&po[0], one(v0));
    dq8::st_stream(&po[hop], one(v1));
    dq8::st_stream(&po[2 * hop], one(v2));
    dq8::st_stream(&po[3 * hop], one(v3));
  }
  for (; r < r_end; r += step, px += hop, po += hop) dq8::st_stream(&po[0], one(px[0]));
}

template <bool SIGNED>
__global__ void __launch_bounds__(kThreads)
dequantize_lastaxis_v4(const uint32_t* __restrict__ q, float4* __restrict__ out,
                       int64_t rows, int nch4, int rows_per_block,
                       const float4* __restrict__ scale,
                       const int4* __restrict__ zp) {
  const int c4 = blockIdx.x * blockDim.x + threadIdx.x;
  if (c4 >= nch4) return;
  const float4 s = scale[c4];
  const int4 z = zp[c4];
  const int64_t r_begin = (int64_t)blockIdx.y * rows_per_block;
  const int64_t r_end = r_begin + rows_per_block < rows ? r_begin + rows_per_block : rows;
  const int64_t step = blockDim.y;
  const int64_t hop = step * nch4;
  int64_t r = r_begin + threadIdx.y;
  const uint32_t* pq = q + r * nch4 + c4;
  float4* po = out + r * nch4 + c4;
  for (; r + 3 * step < r_end; r += 4 * step, pq += 4 * hop, po += 4 * hop) {
    const uint32_t w0 = pq[0], w1 = pq[hop], w2 = pq[2 * hop], w3 = pq[3 * hop];
    dq8::st_stream(&po[0], dequant_word4<SIGNED>(w0, z, s));
    dq8::st_stream(&po[hop], dequant_word4<SIGNED>(w1, z, s));
    dq8::st_stream(&po[2 * hop], dequant_word4<SIGNED>(w2, z, s));
    dq8::st_stream(&po[3 * hop], dequant_word4<SIGNED>(w3, z, s));
  }
  for (; r < r_end; r += step, pq += hop, po += hop)
    dq8::st_stream(&po[0], dequant_word4<SIGNED>(pq[0], z, s));
}

// ------------------------------------- per channel, inner % 4 == 0 (any axis)
// One (outer, channel) row of `inner` contiguous elements per blockIdx.y; one unit per
// thread.  The row index is uniform over the workgroup and stays in 32 bits.
template <int ROUND>
__global__ void __launch_bounds__(kThreads)
quantize_rows_v4(const float4* __restrict__ x, uint32_t* __restrict__ out,
                 unsigned rows, int64_t inner4, unsigned nch,
                 const float* __restrict__ scale,
                 const int32_t* __restrict__ zp, float lo, float hi) {
  const unsigned row = blockIdx.y + blockIdx.z * gridDim.y;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (row >= rows || i >= inner4) return;
  const float4 v = x[(int64_t)row * inner4 + i];
  // The row's parameters stay scalar (the division is cheaper with a uniform divisor)
  // but are fetched after the data load has been issued: a scalar load ahead of it
  // would be waited for, a cold miss per row, before the data load starts.
  __builtin_amdgcn_sched_barrier(0);
  const unsigned c = row % nch;
  const float s = scale[c];
  const float z = (float)zp[c];
  out[(int64_t)row * inner4 + i] =
      divisor_in_fast_range(s)
          ? quant4_by_constant<ROUND>(v, s, 1.0f / s, z, lo, hi)
          : pack4(quant_one<ROUND>(v.x, s, z, lo, hi), quant_one<ROUND>(v.y, s, z, lo, hi),
                  quant_one<ROUND>(v.z, s, z, lo, hi), quant_one<ROUND>(v.w, s, z, lo, hi));
}

// The grid of the row kernels: a workgroup per UNIT * kThreads groups of four of a row.
struct RowsGrid {
  unsigned x, y;
  int64_t z;
};
template <int UNIT>
RowsGrid rows_grid(int64_t rows, int64_t inner4) {
  const unsigned y = (unsigned)std::min<int64_t>(rows, 32768);
  return {(unsigned)dq8::ceil_div(inner4, UNIT * kThreads), y, dq8::ceil_div(rows, y)};
}

// One (outer, channel) row of `inner_words` 4-byte words per blockIdx.y; UNIT words per thread,
// kThreads apart, so that every load and store instruction of a wave is one contiguous span
// (UNIT = 1: 4 bytes in, one 16-byte store; UNIT = 2: two of each).
template <bool SIGNED, int UNIT>
__global__ void __launch_bounds__(kThreads)
dequantize_rows(const uint32_t* __restrict__ q, float4* __restrict__ out,
                unsigned rows, int64_t inner_words, unsigned nch,
                const float* __restrict__ scale, const int32_t* __restrict__ zp) {
  const unsigned row = blockIdx.y + blockIdx.z * gridDim.y;
  if (row >= rows) return;
  const unsigned c = row % nch + opaque_zero();
  const float s = scale[c];
  const int z = zp[c];
  const uint32_t* pq = q + (int64_t)row * inner_words;
  float4* po = out + (int64_t)row * inner_words;
  for (int64_t i = (int64_t)blockIdx.x * (UNIT * kThreads) + threadIdx.x; i < inner_words;
       i += (int64_t)gridDim.x * (UNIT * kThreads)) {
    if (UNIT == 2) {
      const bool two = i + kThreads < inner_words;
      const uint32_t w0 = pq[i];
      const uint32_t w1 = two ? pq[i + kThreads] : 0u;
      dq8::st_stream(&po[i], dequant_word<SIGNED>(w0, z, s));
      if (two) dq8::st_stream(&po[i + kThreads], dequant_word<SIGNED>(w1, z, s));
    } else {
      dq8::st_stream(&po[i], dequant_word<SIGNED>(pq[i], z, s));
    }
  }
}

// ------------------------------------------------------------------ fake quant
template <int ROUND>
__global__ void __launch_bounds__(kThreads)
fake_quant_tensor_v4(const float4* __restrict__ x, float4* __restrict__ out, int64_t n,
                     const float* __restrict__ scale, const int32_t* __restrict__ zp, float lo,
                     float hi) {
  const int64_t n4 = n >> 2;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i < n4) {
    float4 v = x[i];                       // (the data load first, as in quantize_tensor_v4)
    __builtin_amdgcn_sched_barrier(0);
    const float s = scale[0];
    const int z = zp[0];
    const float y = 1.0f / s;
    const bool fast = divisor_in_fast_range(s);
    for (;;) {
      dq8::st_stream(&out[i],
                     fast ? fake4_by_constant<ROUND>(v, s, y, z, lo, hi)
                          : make_float4(fake_one<ROUND>(v.x, s, z, lo, hi), fake_one<ROUND>(v.y, s, z, lo, hi),
                                        fake_one<ROUND>(v.z, s, z, lo, hi), fake_one<ROUND>(v.w, s, z, lo, hi)));
      i += stride;
      if (i >= n4) break;
      v = x[i];
    }
  }
  if (i - n4 < (n & 3)) {                  // the up to three elements behind the last four
    const int64_t e = i + 3 * n4;
    reinterpret_cast<float*>(out)[e] =
        fake_one<ROUND>(reinterpret_cast<const float*>(x)[e], scale[0], zp[0], lo, hi);
  }
}

template <int ROUND>
__global__ void __launch_bounds__(kThreads)
fake_quant_lastaxis_v4(const float4* __restrict__ x, float4* __restrict__ out, int64_t rows,
                       int nch4, int rows_per_block, const float4* __restrict__ scale,
                       const int4* __restrict__ zp, float lo, float hi) {
  const int c4 = blockIdx.x * blockDim.x + threadIdx.x;
  if (c4 >= nch4) return;
  const float4 s = scale[c4];
  const int4 z = zp[c4];
  const int64_t r_begin = (int64_t)blockIdx.y * rows_per_block;
  const int64_t r_end = r_begin + rows_per_block < rows ? r_begin + rows_per_block : rows;
  const int64_t step = blockDim.y;
  const int64_t hop = step * nch4;
  int64_t r = r_begin + threadIdx.y;
  const float4* px = x + r * nch4 + c4;
  float4* po = out + r * nch4 + c4;
  auto one = [&](const float4& v) {
    return make_float4(fake_one<ROUND>(v.x, s.x, z.x, lo, hi), fake_one<ROUND>(v.y, s.y, z.y, lo, hi),
                       fake_one<ROUND>(v.z, s.z, z.z, lo, hi), fake_one<ROUND>(v.w, s.w, z.w, lo, hi));
  };
  for (; r + 3 * step < r_end; r += 4 * step, px += 4 * hop, po += 4 * hop) {
    const float4 v0 = px[0], v1 = px[hop], v2 = px[2 * hop], v3 = px[3 * hop];
    dq8::st_stream(&po[0], one(v0));
    dq8::st_stream(&po[hop], one(v1));
    dq8::st_stream(&po[2 * hop], one(v2));
    dq8::st_stream(&po[3 * hop], one(v3));
  }
  for (; r < r_end; r += step, px += hop, po += hop) dq8::st_stream(&po[0], one(px[0]));
}

template <int ROUND>
__global__ void __launch_bounds__(kThreads)
fake_quant_rows_v4(const float4* __restrict__ x, float4* __restrict__ out, unsigned rows,
                   int64_t inner4, unsigned nch, const float* __restrict__ scale,
                   const int32_t* __restrict__ zp, float lo, float hi) {
  const unsigned row = blockIdx.y + blockIdx.z * gridDim.y;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (row >= rows || i >= inner4) return;
  const float4 v = x[(int64_t)row * inner4 + i];
  __builtin_amdgcn_sched_barrier(0);   // parameters after the data load, as in quantize_rows_v4
  const unsigned c = row % nch;
  const float s = scale[c];
  const int z = zp[c];
  dq8::st_stream(&out[(int64_t)row * inner4 + i],
                 make_float4(fake_one<ROUND>(v.x, s, z, lo, hi), fake_one<ROUND>(v.y, s, z, lo, hi),
                             fake_one<ROUND>(v.z, s, z, lo, hi), fake_one<ROUND>(v.w, s, z, lo, hi)));
}

// ------------------------------------------------- any type, size and alignment
// The conversion of the clamped f32 value saturates: the f32 images of 2^31 - 1 and 2^32 - 1 are
// 2^31 and 2^32, one past the integer range.
template <typename QT>
__device__ __forceinline__ QT convert_clamped(float t) {
  return (QT)(int)t;
}
template <>
__device__ __forceinline__ int32_t convert_clamped<int32_t>(float t) {
  return t >= 2147483648.0f ? INT32_MAX : (int32_t)t;
}
template <>
__device__ __forceinline__ uint32_t convert_clamped<uint32_t>(float t) {
  return t >= 4294967296.0f ? UINT32_MAX : (t <= 0.0f ? 0u : (uint32_t)t);
}
template <>
__device__ __forceinline__ uint16_t convert_clamped<uint16_t>(float t) {
  return (uint16_t)(unsigned)t;
}

// Four elements of a type as one memory operation.
template <typename T>
struct alignas(4 * sizeof(T)) Four {
  T v[4];
};
template <typename T>
__device__ __forceinline__ void st_stream_four(T* p, const Four<T>& f) {
  if constexpr (sizeof(T) == 1) {
    dq8::st_stream(reinterpret_cast<uint32_t*>(p), __builtin_bit_cast(uint32_t, f));
  } else if constexpr (sizeof(T) == 2) {
    __builtin_nontemporal_store(__builtin_bit_cast(uint64_t, f), reinterpret_cast<uint64_t*>(p));
  } else {
    dq8::st_stream(reinterpret_cast<float4*>(p), __builtin_bit_cast(float4, f));
  }
}

template <typename OP, typename IN, typename OUT>
__device__ __forceinline__ void each_of_four(const OP& op, const Four<IN>& x, const float4& s, const int4& z,
                                             Four<OUT>& o) {
  op(x.v[0], s.x, z.x, o.v[0]);
  op(x.v[1], s.y, z.y, o.v[1]);
  op(x.v[2], s.z, z.z, o.v[2]);
  op(x.v[3], s.w, z.w, o.v[3]);
}

// What the general kernels do to one element: XT -> QT quantizes, QT -> float dequantizes,
// float -> float fake-quantizes.
template <int ROUND>
struct Quantize {
  static constexpr bool kByReciprocal = true;      // quick's results are those of the division where it says so
  float lo, hi;
  template <typename XT, typename QT>
  __device__ __forceinline__ void operator()(const XT& x, float s, int z, QT& q) const {
    const float t1 = (float)x / s + (float)z;
    const float t2 = ROUND == DQ8_ROUND_HALF_TO_EVEN ? rintf(t1) : roundf(t1);
    q = convert_clamped<QT>(fminf(fmaxf(t2, lo), hi));
  }
  // four at a time, divided through the reciprocals y, which the divisors have to allow (the quotients'
  // bits are those of the division, see div4_by_constant); false where they don't come out finite
  template <typename XT, typename QT>
  __device__ __forceinline__ bool quick(const Four<XT>& x, const float4& s, const float4& y, const int4& z,
                                        Four<QT>& q) const {
    float4 d;
    const bool ok = div4_quick(make_float4((float)x.v[0], (float)x.v[1], (float)x.v[2], (float)x.v[3]), s, y, d);
    const float t[4] = {d.x + (float)z.x, d.y + (float)z.y, d.z + (float)z.z, d.w + (float)z.w};
    if constexpr (sizeof(QT) == 1 && ROUND == DQ8_ROUND_HALF_TO_EVEN) {
      q = __builtin_bit_cast(Four<QT>, quant4_pack_rne(make_float4(t[0], t[1], t[2], t[3]), lo, hi));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float r = ROUND == DQ8_ROUND_HALF_TO_EVEN ? rintf(t[i]) : roundf(t[i]);
        q.v[i] = convert_clamped<QT>(fminf(fmaxf(r, lo), hi));
      }
    }
    return ok;
  }
};
struct Dequantize {
  static constexpr bool kByReciprocal = false;
  template <typename QT>
  __device__ __forceinline__ void operator()(const QT& q, float s, int z, float& y) const {
    // (the input is converted to the zero point's type, i32, before the subtraction)
    y = (float)((int32_t)q - z) * s;
  }
  template <typename QT>
  __device__ __forceinline__ bool quick(const Four<QT>& q, const float4& s, const float4&, const int4& z,
                                        Four<float>& y) const {
    each_of_four(*this, q, s, z, y);
    return true;
  }
};
template <int ROUND>
struct FakeQuantize {
  static constexpr bool kByReciprocal = false;
  float lo, hi;
  __device__ __forceinline__ void operator()(float x, float s, int z, float& y) const {
    y = fake_one<ROUND>(x, s, z, lo, hi);
  }
  __device__ __forceinline__ bool quick(const Four<float>& x, const float4& s, const float4&, const int4& z,
                                        Four<float>& y) const {
    each_of_four(*this, x, s, z, y);
    return true;
  }
};

__device__ __forceinline__ bool divisors_in_fast_range(const float4& s) {
  return divisor_in_fast_range(s.x) && divisor_in_fast_range(s.y) && divisor_in_fast_range(s.z) &&
         divisor_in_fast_range(s.w);
}

typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef int i4_any __attribute__((ext_vector_type(4), aligned(4)));

// The parameters of channel c < nch and the next three, cyclically.
__device__ __forceinline__ void four_parameters(const float* scale, const int32_t* zp, uint32_t c, uint32_t nch,
                                                float4& s, int4& z) {
  if (c + 3 < nch) {
    const f4_any a = *reinterpret_cast<const f4_any*>(scale + c);
    const i4_any b = *reinterpret_cast<const i4_any*>(zp + c);
    s = make_float4(a.x, a.y, a.z, a.w);
    z = make_int4(b.x, b.y, b.z, b.w);
  } else {
    uint32_t k[4] = {c};
#pragma unroll
    for (int i = 1; i < 4; ++i) k[i] = k[i - 1] + 1 == nch ? 0 : k[i - 1] + 1;
    s = make_float4(scale[k[0]], scale[k[1]], scale[k[2]], scale[k[3]]);
    z = make_int4(zp[k[0]], zp[k[1]], zp[k[2]], zp[k[3]]);
  }
}

// Per channel on the last axis, any number of channels.  Four rows of nch elements are nch groups
// of four, and group u of every such block of rows belongs to the same four channels (4 u mod nch
// and the next three, cyclically), whatever nch: the threads of the [rows, channels] pattern, with
// their scales and zero points in registers, on a tensor whose rows start anywhere.
// Bound: HBM, below a few million elements the launch and one trip to memory -- hence four loads in
// flight, ahead of everything else, and all parameters in two more.  1000 x 3073 to uint8 7.4 us with two
// groups in flight and eight parameter loads, 5.9 so (the even 1000 x 3072: 4.5); 16000 x 3073 57.6 ->
// 44.3, from f16 53.3 -> 29.0 (16000 x 3072: 5.6 TB/s); 8000 x 201 4.8 -> 3.85.
template <typename IN, typename OUT, typename OP>
__global__ void __launch_bounds__(kThreads)
lastaxis_any(const IN* __restrict__ in, OUT* __restrict__ out, int64_t n, int nch, int blocks4,
             int per_thread_block, const float* __restrict__ scale, const int32_t* __restrict__ zp,
             const OP op) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= nch) return;
  const int64_t n4 = n >> 2;
  const int step = blockDim.y;                   // blocks of rows between two of this thread
  const int r_begin = blockIdx.y * per_thread_block + threadIdx.y;
  const int r_end = min((int)(blockIdx.y + 1) * per_thread_block, blocks4);
  // (only in the last block of rows can the group be missing or short)
  const int last = blocks4 - 1;
  const bool whole_last = (int64_t)last * nch + u < n4;
  const int r_whole = whole_last ? r_end : min(r_end, last);
  // Groups in flight, the first ones ahead of the parameters.  Rows past the end are read as the last
  // one: no branch around a load.
  constexpr int U = 4;
  Four<IN> x[U];
  auto fetch = [&](int r) {
#pragma unroll
    for (int k = 0; k < U; ++k)
      x[k] = *reinterpret_cast<const Four<IN>*>(in + 4 * ((int64_t)min(r + k * step, r_whole - 1) * nch + u));
  };
  if (r_begin < r_whole) fetch(r_begin);
  __builtin_amdgcn_sched_barrier(0);
  int c = 4 * u;
#pragma unroll
  for (int i = 0; i < 3; ++i) c -= c >= nch ? nch : 0;
  float4 s;
  int4 z;
  four_parameters(scale, zp, c, nch, s, z);
  const float4 y = make_float4(1.0f / s.x, 1.0f / s.y, 1.0f / s.z, 1.0f / s.w);
  const bool fast = !OP::kByReciprocal || divisors_in_fast_range(s);
  for (int r = r_begin; r < r_whole;) {
    Four<OUT> o[U];
    bool ok = fast;
#pragma unroll
    for (int k = 0; k < U; ++k) ok &= op.quick(x[k], s, y, z, o[k]);
    OUT* const po = out + 4 * ((int64_t)r * nch + u);
    const int64_t hop = 4 * (int64_t)step * nch;
    if (__builtin_expect(ok, 1)) {
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (r + k * step < r_whole) st_stream_four(po + k * hop, o[k]);
    } else {
      // (one copy of the divisions for all groups: inlined behind each they were 12 KiB of code that
      // every wave of a launch fetched, 16 us)
#pragma unroll 1
      for (int k = 0; k < U; ++k) {
        Four<IN> v = x[0];
#pragma unroll
        for (int j = 1; j < U; ++j)
          if (j == k) v = x[j];
        Four<OUT> w;
        each_of_four(op, v, s, z, w);
        if (r + k * step < r_whole) st_stream_four(po + k * hop, w);
      }
    }
    r += U * step;
    if (r < r_whole) fetch(r);
  }
  const int64_t g = (int64_t)last * nch + u;
  if (g == n4 && r_end == blocks4 && ((last - r_begin) & (step - 1)) == 0 && last >= r_begin) {
    const float st[3] = {s.x, s.y, s.z};         // the up to three elements behind the last four
    const int zt[3] = {z.x, z.y, z.z};
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (4 * n4 + i < n) op(in[4 * n4 + i], st[i], zt[i], out[4 * n4 + i]);
  }
}

// One linear sweep, n < 2^32: a workgroup takes U chunks of kThreads groups of four, kHop groups apart.
// PER_CHANNEL: the channels on the last axis, a group's parameters read with it (advance = 4 kHop mod nch);
// otherwise per tensor.
// Bound: HBM.  U: 16 KiB of f32 or 8 KiB of a narrower type on their way per workgroup, less where the
// results are 4 bytes wide and as many stores follow the loads (four instead of two or one: 2-5 % slower
// on large tensors).  Us, 16000 x 3072 per tensor: f16 to uint8 44.0 -> 23.6 (6.2 TB/s) with one load of 8
// bytes per thread before, f16 to int16 48.3 -> 31.0, f32 to int16 54.5 -> 50.7; 16000 x 3073 by channel:
// uint8 to f32 51.5 -> 35.5, fake quantization 74.1 -> 69.2; 1000 x 3073 6.7 -> 4.0 and 7.6 -> 5.7.
template <typename IN, typename OUT, typename OP, bool PER_CHANNEL, int U>
__global__ void __launch_bounds__(kThreads)
sweep_any(const IN* __restrict__ in, OUT* __restrict__ out, uint32_t n, uint32_t nch, uint32_t advance,
          const float* __restrict__ scale, const int32_t* __restrict__ zp, const OP op) {
  constexpr int P = PER_CHANNEL ? U : 1;
  const uint32_t n4 = n >> 2;
  const uint32_t g0 = sweep_first_group<U>();
  if (g0 > n4) return;
  Four<IN> x[U];
#pragma unroll
  for (int k = 0; k < U; ++k)                    // (groups past the end are read as the last one)
    x[k] = *reinterpret_cast<const Four<IN>*>(in + 4 * (size_t)min(g0 + k * kHop, n4 - 1));
  __builtin_amdgcn_sched_barrier(0);
  float4 s[P];
  int4 z[P];
  if constexpr (PER_CHANNEL) {
    uint32_t c = (4 * g0) % nch;
#pragma unroll
    for (int k = 0; k < P; ++k) {
      four_parameters(scale, zp, c, nch, s[k], z[k]);
      c += advance;
      c -= c >= nch ? nch : 0;
    }
  } else {
    const float s1 = scale[0];
    const int z1 = zp[0];
    s[0] = make_float4(s1, s1, s1, s1);
    z[0] = make_int4(z1, z1, z1, z1);
  }
  Four<OUT> o[U];
  bool ok = true;
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const float4& sk = s[k % P];
    if (OP::kByReciprocal) ok &= divisors_in_fast_range(sk);
    const float4 y = make_float4(1.0f / sk.x, 1.0f / sk.y, 1.0f / sk.z, 1.0f / sk.w);
    ok &= op.quick(x[k], sk, y, z[k % P], o[k]);
  }
  if (__builtin_expect(ok, 1)) {
#pragma unroll
    for (int k = 0; k < U; ++k)
      if (g0 + k * kHop < n4) st_stream_four(out + 4 * (size_t)(g0 + k * kHop), o[k]);
  } else {                                       // (one copy of the divisions, as in lastaxis_any)
#pragma unroll 1
    for (int k = 0; k < U; ++k) {
      Four<IN> v = x[0];
      float4 sk = s[0];
      int4 zk = z[0];
#pragma unroll
      for (int j = 1; j < U; ++j)
        if (j == k) {
          v = x[j];
          sk = s[j % P];
          zk = z[j % P];
        }
      Four<OUT> w;
      each_of_four(op, v, sk, zk, w);
      if (g0 + k * kHop < n4) st_stream_four(out + 4 * (size_t)(g0 + k * kHop), w);
    }
  }
  if ((n & 3) != 0 && (n4 - g0) % kHop == 0 && n4 - g0 < U * kHop) {
    // the up to three elements behind the last four
    for (uint32_t e = 4 * n4; e < n; ++e) {
      const uint32_t c = PER_CHANNEL ? e % nch : 0;
      op(in[e], scale[c], zp[c], out[e]);
    }
  }
}

// The same sweep with the channel on another axis, rows of inner >= 4 elements: a group of four lies in
// one row or across the end of one.  16000 x 3072, a channel a row, f16 to uint8 55.6 -> 31.5 us, f32 to
// int16 61.1 -> 50.7 and back 55.3 -> 46.4; 16000 x 3073 to uint8 55.9 -> 42.0, 1000 x 3073 6.1 -> 5.15.
// A workgroup's groups follow each other here, in pieces of 1024 groups whatever U, piece j on die j % 8
// (the 4 / U workgroups of a piece are eight apart): kHop apart, f16 to uint8 in buffers that change took
// 10.0-10.6 us at 4000 x 3072 in place of 9.55.
template <int U>
__device__ __forceinline__ uint32_t piece_first_group() {
  constexpr uint32_t R = 4 / U;
  const uint32_t b = blockIdx.x, piece = b / (8 * R) * 8 + b % 8, part = b / 8 % R;
  return piece * (4 * kThreads) + part * (U * kThreads) + threadIdx.x;
}
template <int U>
unsigned piece_workgroups(int64_t n) {           // (one group more: the elements behind the last four)
  const int64_t pieces = dq8::ceil_div(n / 4 + 1, (int64_t)(4 * kThreads));
  return (unsigned)(U == 4 ? pieces : dq8::ceil_div(pieces, 8) * 8 * (4 / U));
}
template <typename IN, typename OUT, typename OP, int U>
__global__ void __launch_bounds__(kThreads)
rows_any(const IN* __restrict__ in, OUT* __restrict__ out, uint32_t n, uint32_t nch, uint32_t inner,
         const float* __restrict__ scale, const int32_t* __restrict__ zp, const OP op) {
  const uint32_t n4 = n >> 2;
  const uint32_t g0 = piece_first_group<U>();
  if (g0 > n4) return;
  Four<IN> x[U];
#pragma unroll
  for (int k = 0; k < U; ++k)                    // (groups past the end are read as the last one)
    x[k] = *reinterpret_cast<const Four<IN>*>(in + 4 * (size_t)min(g0 + k * kThreads, n4 - 1));
  __builtin_amdgcn_sched_barrier(0);
  // the row's channel and the element's place in it
  const uint32_t row = 4 * g0 / inner;
  uint32_t at = 4 * g0 - row * inner, c = row % nch;
  float s0[U], s1[U];
  int z0[U], z1[U];
  uint32_t left[U];                              // elements of the row from the group's first one on
#pragma unroll
  for (int k = 0; k < U; ++k) {
    left[k] = inner - at;
    const uint32_t next = left[k] >= 4 ? c : c + 1 == nch ? 0 : c + 1;
    s0[k] = scale[c];
    z0[k] = zp[c];
    s1[k] = scale[next];
    z1[k] = zp[next];
    at += 4 * kThreads;
    if (at >= inner) {
      const uint32_t rows = inner >= 4 * kThreads ? 1 : at / inner;
      at -= rows * inner;
      c += rows;
      if (c >= nch) c = c - nch < nch ? c - nch : c % nch;
    }
  }
  auto parameters = [&](int k, float4& s, int4& z) {
    const bool b = left[k] < 2, d = left[k] < 3, e = left[k] < 4;
    s = make_float4(s0[k], b ? s1[k] : s0[k], d ? s1[k] : s0[k], e ? s1[k] : s0[k]);
    z = make_int4(z0[k], b ? z1[k] : z0[k], d ? z1[k] : z0[k], e ? z1[k] : z0[k]);
  };
  Four<OUT> o[U];
  bool ok = true;
#pragma unroll
  for (int k = 0; k < U; ++k) {
    float4 s;
    int4 z;
    parameters(k, s, z);
    const float y0 = 1.0f / s0[k], y1 = 1.0f / s1[k];
    if (OP::kByReciprocal) ok &= divisor_in_fast_range(s0[k]) && divisor_in_fast_range(s1[k]);
    const float4 y = make_float4(y0, left[k] < 2 ? y1 : y0, left[k] < 3 ? y1 : y0, left[k] < 4 ? y1 : y0);
    ok &= op.quick(x[k], s, y, z, o[k]);
  }
  if (__builtin_expect(ok, 1)) {
#pragma unroll
    for (int k = 0; k < U; ++k)
      if (g0 + k * kThreads < n4) st_stream_four(out + 4 * (size_t)(g0 + k * kThreads), o[k]);
  } else {                                       // (one copy of the divisions, as in lastaxis_any)
#pragma unroll 1
    for (int k = 0; k < U; ++k) {
      Four<IN> v = x[0];
      float4 s, sj;
      int4 z, zj;
      parameters(0, s, z);
#pragma unroll
      for (int j = 1; j < U; ++j) {
        parameters(j, sj, zj);
        if (j == k) {
          v = x[j];
          s = sj;
          z = zj;
        }
      }
      Four<OUT> w;
      each_of_four(op, v, s, z, w);
      if (g0 + k * kThreads < n4) st_stream_four(out + 4 * (size_t)(g0 + k * kThreads), w);
    }
  }
  if ((n & 3) != 0 && (n4 - g0) % kThreads == 0 && n4 - g0 < U * kThreads) {
    // the up to three elements behind the last four
    for (uint32_t e = 4 * n4; e < n; ++e) {
      const uint32_t ce = e / inner % nch;
      op(in[e], scale[ce], zp[ce], out[e]);
    }
  }
}

// Any axis (or per tensor): four consecutive elements per thread, whose channels follow from the
// first one's by counting on.  VEC: the four are one memory operation.  INDEX: wide enough for n.
template <typename IN, typename OUT, typename OP, bool VEC, typename INDEX>
__global__ void __launch_bounds__(kThreads)
flat_any(const IN* __restrict__ in, OUT* __restrict__ out, int64_t n, int64_t nch, int64_t inner,
         int per_channel, const float* __restrict__ scale, const int32_t* __restrict__ zp, const OP op) {
  const int64_t first = 4 * ((int64_t)blockIdx.x * kThreads + threadIdx.x);
  if (first >= n) return;
  const int left = n - first < 4 ? (int)(n - first) : 4;
  Four<IN> x;
  if (VEC && left == 4) {
    x = *reinterpret_cast<const Four<IN>*>(in + first);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < left) x.v[i] = in[first + i];
  }
  // (the parameters after the data load has been issued)
  float sv[4];
  int zv[4];
  if (!per_channel) {
    sv[0] = sv[1] = sv[2] = sv[3] = scale[0];
    zv[0] = zv[1] = zv[2] = zv[3] = zp[0];
  } else {
    const INDEX row = (INDEX)first / (INDEX)inner;
    INDEX at = (INDEX)first - row * (INDEX)inner, c = row % (INDEX)nch;
    sv[0] = scale[c];
    zv[0] = zp[c];
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      sv[i] = sv[i - 1];
      zv[i] = zv[i - 1];
      if (++at == (INDEX)inner && i < left) {
        at = 0;
        c = c + 1 == (INDEX)nch ? 0 : c + 1;
        sv[i] = scale[c];
        zv[i] = zp[c];
      }
    }
  }
  if (VEC && left == 4) {
    const float4 s = make_float4(sv[0], sv[1], sv[2], sv[3]);
    const int4 z = make_int4(zv[0], zv[1], zv[2], zv[3]);
    Four<OUT> o;
    if (!divisors_in_fast_range(s) ||
        !op.quick(x, s, make_float4(1.0f / s.x, 1.0f / s.y, 1.0f / s.z, 1.0f / s.w), z, o))
      each_of_four(op, x, s, z, o);
    st_stream_four(out + first, o);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < left) op(x.v[i], sv[i], zv[i], out[first + i]);
  }
}

inline bool sweep_takes(int64_t n) { return n >= 4 && n < (1LL << 32) - 131072; }
template <bool PER_CHANNEL, typename IN, typename OUT, typename OP>
int launch_sweep(const IN* in, OUT* out, int64_t n, int64_t nch, const float* scale, const int32_t* zp, const OP& op,
                 hipStream_t st) {
  constexpr int U = sizeof(OUT) < 4 ? 4 : PER_CHANNEL ? 2 : sizeof(IN) < 4 ? 2 : 1;
  hipLaunchKernelGGL((sweep_any<IN, OUT, OP, PER_CHANNEL, U>), dim3(sweep_workgroups<U>(n)),
                     dim3(kThreads), 0, st, in, out, (uint32_t)n, (uint32_t)nch, (uint32_t)(4 * kHop % nch), scale,
                     zp, op);
  return dq8::check_hip(hipGetLastError(), "quantize / dequantize launch");
}

template <typename IN, typename OUT, typename OP>
int launch_any(const IN* in, OUT* out, int64_t outer, int64_t nch, int64_t inner, bool per_channel,
               const float* scale, const int32_t* zp, const OP& op, hipStream_t st) {
  const int64_t n = outer * nch * inner;
  const bool vec = dq8::aligned(in, sizeof(Four<IN>)) && dq8::aligned(out, sizeof(Four<OUT>));
  if (vec && per_channel && inner == 1 && outer >= 4 && nch < (1 << 28)) {
    const int64_t blocks4 = dq8::ceil_div(outer, 4);          // four rows each, the last perhaps fewer
    const LastAxisPlan lp = plan_last_axis(blocks4, (int)nch);
    // The sweep reads the parameters with every group, and its wave instructions cover whole lines; the
    // rows keep the parameters, but start at any 16 bytes, which costs little for reads and narrow
    // results and a third for 4-byte ones.  us, rows / sweep, dequantize uint8: 16000 x 3073 48.0 /
    // 35.5, 1000 x 1025 3.83 / 2.97, 8000 x 201 3.55 / 3.92; quantize to uint8: 44.5 / 50.0, 3.73 / 3.61,
    // 3.84 / 4.55, and 5.77 / 4.70 at 8000 x 257, where half the threads of the rows have no channel.
    const bool sweep = sizeof(OUT) == 4 ? nch >= kThreads : nch >= kThreads && 4 * (int64_t)lp.gx * lp.bx > 5 * nch;
    if (sweep && sweep_takes(n))
      return launch_sweep<true>(in, out, n, nch, scale, zp, op, st);
    if (blocks4 < (1LL << 30)) {
      hipLaunchKernelGGL((lastaxis_any<IN, OUT, OP>), dim3(lp.gx, lp.gy), dim3(lp.bx, lp.by), 0, st, in, out, n,
                         (int)nch, (int)blocks4, lp.rows_per_block, scale, zp, op);
      return dq8::check_hip(hipGetLastError(), "quantize / dequantize launch");
    }
  }
  if (vec && !per_channel && sweep_takes(n)) return launch_sweep<false>(in, out, n, 1, scale, zp, op, st);
  // (narrow results of few elements: four groups a thread leave too few workgroups, 30000 x 37 to int16 3.80
  // against 3.47 us, 100 x 500 3.14 against 2.52; from 1.5 M on the sweep wins, 4000 x 513 3.9 against 4.3)
  if (vec && per_channel && inner >= 4 && sweep_takes(n) && (sizeof(OUT) == 4 || n >= 1500000)) {
    constexpr int U = sizeof(OUT) < 4 ? 4 : sizeof(IN) < 4 ? 2 : 1;
    hipLaunchKernelGGL((rows_any<IN, OUT, OP, U>), dim3(piece_workgroups<U>(n)),
                       dim3(kThreads), 0, st, in, out, (uint32_t)n, (uint32_t)nch, (uint32_t)inner, scale, zp, op);
    return dq8::check_hip(hipGetLastError(), "quantize / dequantize launch");
  }
  const int64_t groups = dq8::ceil_div(n, 4 * (int64_t)kThreads);
  DQ8_REQUIRE(groups < (1LL << 31), "quantize / dequantize: tensor too large for one launch");
  auto kern = n < (1LL << 32) - 4 ? (vec ? flat_any<IN, OUT, OP, true, uint32_t> : flat_any<IN, OUT, OP, false, uint32_t>)
                                  : (vec ? flat_any<IN, OUT, OP, true, uint64_t> : flat_any<IN, OUT, OP, false, uint64_t>);
  hipLaunchKernelGGL(kern, dim3((unsigned)groups), dim3(kThreads), 0, st, in, out, n, nch, inner,
                     (int)per_channel, scale, zp, op);
  return dq8::check_hip(hipGetLastError(), "quantize / dequantize launch");
}

template <typename XT, typename QT>
int launch_quantize_any(bool rne, const XT* x, void* out, int64_t outer, int64_t nch, int64_t inner,
                        bool per_channel, const float* scale, const int32_t* zp, float lo, float hi,
                        hipStream_t st) {
  return rne ? launch_any(x, static_cast<QT*>(out), outer, nch, inner, per_channel, scale, zp,
                          Quantize<DQ8_ROUND_HALF_TO_EVEN>{lo, hi}, st)
             : launch_any(x, static_cast<QT*>(out), outer, nch, inner, per_channel, scale, zp,
                          Quantize<DQ8_ROUND_HALF_AWAY_FROM_ZERO>{lo, hi}, st);
}

template <typename XT>
int launch_quantize_kind(int out_kind, bool rne, const XT* x, void* out, int64_t outer, int64_t nch,
                         int64_t inner, bool per_channel, const float* scale, const int32_t* zp,
                         float lo, float hi, hipStream_t st) {
#define DQ8_KIND_CASE(KIND, QT) \
  case KIND:                    \
    return launch_quantize_any<XT, QT>(rne, x, out, outer, nch, inner, per_channel, scale, zp, lo, hi, st);
  switch (out_kind) {
    DQ8_KIND_CASE(DQ8_I8, int8_t)
    DQ8_KIND_CASE(DQ8_U8, uint8_t)
    DQ8_KIND_CASE(DQ8_I16, int16_t)
    DQ8_KIND_CASE(DQ8_U16, uint16_t)
    DQ8_KIND_CASE(DQ8_I32, int32_t)
    DQ8_KIND_CASE(DQ8_U32, uint32_t)
  }
#undef DQ8_KIND_CASE
  return dq8::fail("quantize: unknown out_kind");
}

}  // namespace

extern "C" int dq8_quantize(const float* x, void* out, int out_kind,
                            int64_t outer, int64_t nch, int64_t inner,
                            const float* scale, const int32_t* zp, int64_t n_q,
                            int32_t qmin, int32_t qmax, int round_mode,
                            void* stream) {
  dq8::clear_error();
  DQ8_REQUIRE(outer >= 0 && nch >= 0 && inner >= 0, "dq8_quantize: negative size");
  DQ8_REQUIRE(out_kind == DQ8_I8 || out_kind == DQ8_U8,
              "dq8_quantize: out_kind must be DQ8_I8 or DQ8_U8");
  DQ8_REQUIRE(round_mode == DQ8_ROUND_HALF_TO_EVEN ||
                  round_mode == DQ8_ROUND_HALF_AWAY_FROM_ZERO,
              "dq8_quantize: unknown round_mode");
  DQ8_REQUIRE(n_q == 1 || n_q == nch, "dq8_quantize: n_q must be 1 or nch");
  const int lim_lo = out_kind == DQ8_I8 ? -128 : 0;
  const int lim_hi = out_kind == DQ8_I8 ? 127 : 255;
  DQ8_REQUIRE(qmin <= qmax && qmin >= lim_lo && qmax <= lim_hi,
              "dq8_quantize: quant_min/quant_max outside the output type");
  const int64_t n = outer * nch * inner;
  if (n == 0) return 0;
  DQ8_REQUIRE(x && out && scale && zp, "dq8_quantize: null pointer");
  hipStream_t st = (hipStream_t)stream;
  const float lo = (float)qmin, hi = (float)qmax;
  const bool per_channel = n_q > 1;
  const bool vec_ok = dq8::aligned(x, 16) && dq8::aligned(out, 4);
  const bool rne = round_mode == DQ8_ROUND_HALF_TO_EVEN;
  // (the kernels divide through the reciprocal, 7 vector instructions per element instead of 19:
  // [4096,768] 3.85 -> 3.3 us, [32,56,56,64] 5.7 -> 4.5 us, [65536,4096] 222-226 -> 216 us)

#define LAUNCH_RND(kernel, grid, block, ...)                                        \
  do {                                                                              \
    if (rne)                                                                        \
      hipLaunchKernelGGL((kernel<DQ8_ROUND_HALF_TO_EVEN>), grid, block, 0, st,      \
                         __VA_ARGS__);                                              \
    else                                                                            \
      hipLaunchKernelGGL((kernel<DQ8_ROUND_HALF_AWAY_FROM_ZERO>), grid, block, 0,   \
                         st, __VA_ARGS__);                                          \
  } while (0)

  if (!per_channel && vec_ok) {
    LAUNCH_RND(quantize_tensor_v4, dim3(sweep_grid(n / 4 + n % 4)), dim3(kThreads),
               (const float4*)x, (uint32_t*)out, n, scale, zp, lo, hi);
  } else if (per_channel && vec_ok && inner == 1 && nch % 4 == 0 && nch / 4 < (1 << 30) &&
             dq8::aligned(scale, 16) && dq8::aligned(zp, 16)) {
    const int nch4 = (int)(nch / 4);
    const LastAxisPlan lp = plan_last_axis(outer, nch4);
    LAUNCH_RND(quantize_lastaxis_v4, dim3(lp.gx, lp.gy), dim3(lp.bx, lp.by), (const float4*)x,
               (uint32_t*)out, outer, nch4, lp.rows_per_block, (const float4*)scale,
               (const int4*)zp, lo, hi);
  } else if (per_channel && vec_ok && inner % 4 == 0 && outer * nch < (1LL << 31)) {
    const int64_t rows = outer * nch;
    const int64_t inner4 = inner / 4;
    DQ8_REQUIRE(inner4 < (1LL << 38), "dq8_quantize: rows too long for one launch");
    const RowsGrid g = rows_grid<1>(rows, inner4);
    DQ8_REQUIRE(g.z <= 65535, "dq8_quantize: too many rows for one launch");
    LAUNCH_RND(quantize_rows_v4, dim3(g.x, g.y, (unsigned)g.z), dim3(kThreads),
               (const float4*)x, (uint32_t*)out, (unsigned)rows, inner4, (unsigned)nch, scale,
               zp, lo, hi);
  } else {
    return launch_quantize_kind<float>(out_kind, rne, x, out, outer, nch, inner, per_channel, scale,
                                       zp, lo, hi, st);
  }
#undef LAUNCH_RND
  return dq8::check_hip(hipGetLastError(), "dq8_quantize launch");
}

extern "C" int dq8_dequantize(const void* q, int in_kind, float* out,
                              int64_t outer, int64_t nch, int64_t inner,
                              const float* scale, const int32_t* zp,
                              int64_t n_q, void* stream) {
  dq8::clear_error();
  DQ8_REQUIRE(outer >= 0 && nch >= 0 && inner >= 0, "dq8_dequantize: negative size");
  DQ8_REQUIRE(in_kind == DQ8_I8 || in_kind == DQ8_U8,
              "dq8_dequantize: in_kind must be DQ8_I8 or DQ8_U8");
  DQ8_REQUIRE(n_q == 1 || n_q == nch, "dq8_dequantize: n_q must be 1 or nch");
  const int64_t n = outer * nch * inner;
  if (n == 0) return 0;
  DQ8_REQUIRE(q && out && scale && zp, "dq8_dequantize: null pointer");
  hipStream_t st = (hipStream_t)stream;
  const int is_signed = in_kind == DQ8_I8;
  const bool per_channel = n_q > 1;
  const bool vec_ok = dq8::aligned(q, 4) && dq8::aligned(out, 16);

  if (!per_channel && vec_ok) {
    const bool hops = l2s_hold(n);
    auto k = is_signed ? (hops ? dequantize_tensor_v4x2<true, kHop> : dequantize_tensor_v4x2<true, kThreads>)
                       : (hops ? dequantize_tensor_v4x2<false, kHop> : dequantize_tensor_v4x2<false, kThreads>);
    hipLaunchKernelGGL(k, dim3(hops ? sweep_workgroups<2>(n) : sweep_grid(dq8::ceil_div(n / 4, 2))), dim3(kThreads),
                       0, st, (const uint32_t*)q, (float4*)out, n, scale, zp);
  } else if (per_channel && vec_ok && inner == 1 && nch % 4 == 0 && nch / 4 < (1 << 30) &&
             dq8::aligned(scale, 16) && dq8::aligned(zp, 16)) {
    const int nch4 = (int)(nch / 4);
    const LastAxisPlan lp = plan_last_axis(outer, nch4);
    auto k = is_signed ? dequantize_lastaxis_v4<true> : dequantize_lastaxis_v4<false>;
    hipLaunchKernelGGL(k, dim3(lp.gx, lp.gy), dim3(lp.bx, lp.by), 0, st, (const uint32_t*)q,
                       (float4*)out, outer, nch4, lp.rows_per_block, (const float4*)scale,
                       (const int4*)zp);
  } else if (per_channel && vec_ok && inner % 4 == 0 && outer * nch < (1LL << 31)) {
    const int64_t rows = outer * nch;
    // Two words per thread once a row is several workgroups -- except where one, on quantize's grid, keeps
    // the words on the die that has just written them.  Both in one buffer, two words / one: 1000 x 3072
    // 12.2 / 9.2 us, 1500 x 3072 16.4 / 9.5, 5000 x 3072 29.9 / 26.8, 12000 x 2048 41.5 / 40.3; dequantize alone
    // 4.9 / 4.7, 5.5 / 5.4, 12.7 / 12.1, 18.3 / 18.0 in buffers that change.
    const bool two = inner >= 2048 && !l2s_hold(n);
    const int64_t units = inner / 4;
    RowsGrid g = two ? rows_grid<2>(rows, units) : rows_grid<1>(rows, units);
    g.x = std::min(g.x, 65536u);
    DQ8_REQUIRE(g.z <= 65535, "dq8_dequantize: too many rows for one launch");
    auto k = two ? (is_signed ? dequantize_rows<true, 2> : dequantize_rows<false, 2>)
                 : (is_signed ? dequantize_rows<true, 1> : dequantize_rows<false, 1>);
    hipLaunchKernelGGL(k, dim3(g.x, g.y, (unsigned)g.z), dim3(kThreads), 0, st,
                       (const uint32_t*)q, (float4*)out, (unsigned)rows, units, (unsigned)nch,
                       scale, zp);
  } else {
    return is_signed ? launch_any((const int8_t*)q, out, outer, nch, inner, per_channel, scale, zp,
                                  Dequantize{}, st)
                     : launch_any((const uint8_t*)q, out, outer, nch, inner, per_channel, scale, zp,
                                  Dequantize{}, st);
  }
  return dq8::check_hip(hipGetLastError(), "dq8_dequantize launch");
}

extern "C" int dq8_fake_quant(const float* x, float* out, int64_t outer, int64_t nch,
                              int64_t inner, const float* scale, const int32_t* zp, int64_t n_q,
                              int32_t qmin, int32_t qmax, int round_mode, void* stream) {
  dq8::clear_error();
  DQ8_REQUIRE(outer >= 0 && nch >= 0 && inner >= 0, "dq8_fake_quant: negative size");
  DQ8_REQUIRE(round_mode == DQ8_ROUND_HALF_TO_EVEN ||
                  round_mode == DQ8_ROUND_HALF_AWAY_FROM_ZERO,
              "dq8_fake_quant: unknown round_mode");
  DQ8_REQUIRE(n_q == 1 || n_q == nch, "dq8_fake_quant: n_q must be 1 or nch");
  DQ8_REQUIRE(qmin <= qmax && qmin >= -32768 && qmax <= 65535,
              "dq8_fake_quant: quant_min/quant_max outside the 8- and 16-bit ranges");
  const int64_t n = outer * nch * inner;
  if (n == 0) return 0;
  DQ8_REQUIRE(x && out && scale && zp, "dq8_fake_quant: null pointer");
  hipStream_t st = (hipStream_t)stream;
  const float lo = (float)qmin, hi = (float)qmax;
  const bool per_channel = n_q > 1;
  const bool vec_ok = dq8::aligned(x, 16) && dq8::aligned(out, 16);
  const bool rne = round_mode == DQ8_ROUND_HALF_TO_EVEN;

#define LAUNCH_RND(kernel, grid, block, ...)                                        \
  do {                                                                              \
    if (rne)                                                                        \
      hipLaunchKernelGGL((kernel<DQ8_ROUND_HALF_TO_EVEN>), grid, block, 0, st,      \
                         __VA_ARGS__);                                              \
    else                                                                            \
      hipLaunchKernelGGL((kernel<DQ8_ROUND_HALF_AWAY_FROM_ZERO>), grid, block, 0,   \
                         st, __VA_ARGS__);                                          \
  } while (0)

  if (!per_channel && vec_ok) {
    LAUNCH_RND(fake_quant_tensor_v4, dim3(sweep_grid(n / 4 + n % 4)), dim3(kThreads), (const float4*)x,
               (float4*)out, n, scale, zp, lo, hi);
  } else if (per_channel && vec_ok && inner == 1 && nch % 4 == 0 && nch / 4 < (1 << 30) &&
             dq8::aligned(scale, 16) && dq8::aligned(zp, 16)) {
    const int nch4 = (int)(nch / 4);
    const LastAxisPlan lp = plan_last_axis(outer, nch4);
    LAUNCH_RND(fake_quant_lastaxis_v4, dim3(lp.gx, lp.gy), dim3(lp.bx, lp.by), (const float4*)x,
               (float4*)out, outer, nch4, lp.rows_per_block, (const float4*)scale,
               (const int4*)zp, lo, hi);
  } else if (per_channel && vec_ok && inner % 4 == 0 && outer * nch < (1LL << 31) &&
             inner / 4 < (1LL << 38) && dq8::ceil_div(outer * nch, 32768) <= 65535) {
    const int64_t rows = outer * nch;
    const int64_t inner4 = inner / 4;
    const unsigned gx = (unsigned)dq8::ceil_div(inner4, kThreads);
    const int gy = (int)std::min<int64_t>(rows, 32768);
    const int64_t gz = dq8::ceil_div(rows, gy);
    LAUNCH_RND(fake_quant_rows_v4, dim3(gx, gy, (unsigned)gz), dim3(kThreads), (const float4*)x,
               (float4*)out, (unsigned)rows, inner4, (unsigned)nch, scale, zp, lo, hi);
  } else {
    return rne ? launch_any(x, out, outer, nch, inner, per_channel, scale, zp,
                            FakeQuantize<DQ8_ROUND_HALF_TO_EVEN>{lo, hi}, st)
               : launch_any(x, out, outer, nch, inner, per_channel, scale, zp,
                            FakeQuantize<DQ8_ROUND_HALF_AWAY_FROM_ZERO>{lo, hi}, st);
  }
#undef LAUNCH_RND
  return dq8::check_hip(hipGetLastError(), "dq8_fake_quant launch");
}

namespace {
bool quant_limits(int kind, int64_t* lo, int64_t* hi) {
  switch (kind) {
    case DQ8_I8: *lo = -128; *hi = 127; return true;
    case DQ8_U8: *lo = 0; *hi = 255; return true;
    case DQ8_I16: *lo = -32768; *hi = 32767; return true;
    case DQ8_U16: *lo = 0; *hi = 65535; return true;
    case DQ8_I32: *lo = INT32_MIN; *hi = INT32_MAX; return true;
    case DQ8_U32: *lo = 0; *hi = UINT32_MAX; return true;
  }
  return false;
}
}  // namespace

extern "C" int dq8_quantize_ex(const void* x, int x_dtype, void* out, int out_kind, int64_t outer,
                               int64_t nch, int64_t inner, const float* scale,
                               const int32_t* zp, int64_t n_q, int64_t qmin, int64_t qmax,
                               int round_mode, void* stream) {
  dq8::clear_error();
  int64_t lim_lo = 0, lim_hi = 0;
  DQ8_REQUIRE(quant_limits(out_kind, &lim_lo, &lim_hi), "dq8_quantize_ex: unknown out_kind");
  DQ8_REQUIRE(x_dtype == DQ8_DTYPE_F32 || x_dtype == DQ8_DTYPE_F16,
              "dq8_quantize_ex: input must be f32 or f16");
  DQ8_REQUIRE(qmin <= qmax && qmin >= lim_lo && qmax <= lim_hi,
              "dq8_quantize_ex: quant_min/quant_max outside the output type");
  // f32 -> 8 bit: the bandwidth-tuned kernels
  if (x_dtype == DQ8_DTYPE_F32 && (out_kind == DQ8_I8 || out_kind == DQ8_U8))
    return dq8_quantize(static_cast<const float*>(x), out, out_kind, outer, nch, inner, scale, zp,
                        n_q, (int32_t)qmin, (int32_t)qmax, round_mode, stream);
  DQ8_REQUIRE(outer >= 0 && nch >= 0 && inner >= 0, "dq8_quantize_ex: negative size");
  DQ8_REQUIRE(round_mode == DQ8_ROUND_HALF_TO_EVEN ||
                  round_mode == DQ8_ROUND_HALF_AWAY_FROM_ZERO,
              "dq8_quantize_ex: unknown round_mode");
  DQ8_REQUIRE(n_q == 1 || n_q == nch, "dq8_quantize_ex: n_q must be 1 or nch");
  const int64_t n = outer * nch * inner;
  if (n == 0) return 0;
  DQ8_REQUIRE(x && out && scale && zp, "dq8_quantize_ex: null pointer");
  const bool rne = round_mode == DQ8_ROUND_HALF_TO_EVEN;
  const float lo = (float)qmin, hi = (float)qmax;
  hipStream_t st = (hipStream_t)stream;
  return x_dtype == DQ8_DTYPE_F32
             ? launch_quantize_kind(out_kind, rne, static_cast<const float*>(x), out, outer, nch, inner,
                                    n_q > 1, scale, zp, lo, hi, st)
             : launch_quantize_kind(out_kind, rne, static_cast<const _Float16*>(x), out, outer, nch,
                                    inner, n_q > 1, scale, zp, lo, hi, st);
}

extern "C" int dq8_dequantize_ex(const void* q, int in_kind, float* out, int64_t outer,
                                 int64_t nch, int64_t inner, const float* scale,
                                 const int32_t* zp, int64_t n_q, void* stream) {
  if (in_kind == DQ8_I8 || in_kind == DQ8_U8)
    return dq8_dequantize(q, in_kind, out, outer, nch, inner, scale, zp, n_q, stream);
  dq8::clear_error();
  DQ8_REQUIRE(in_kind >= DQ8_I16 && in_kind <= DQ8_U32, "dq8_dequantize_ex: unknown in_kind");
  DQ8_REQUIRE(outer >= 0 && nch >= 0 && inner >= 0, "dq8_dequantize_ex: negative size");
  DQ8_REQUIRE(n_q == 1 || n_q == nch, "dq8_dequantize_ex: n_q must be 1 or nch");
  const int64_t n = outer * nch * inner;
  if (n == 0) return 0;
  DQ8_REQUIRE(q && out && scale && zp, "dq8_dequantize_ex: null pointer");
  hipStream_t st = (hipStream_t)stream;
#define DQ8_KIND_CASE(QT) \
  launch_any(static_cast<const QT*>(q), out, outer, nch, inner, n_q > 1, scale, zp, Dequantize{}, st)
  switch (in_kind) {
    case DQ8_I16: return DQ8_KIND_CASE(int16_t);
    case DQ8_U16: return DQ8_KIND_CASE(uint16_t);
    case DQ8_I32: return DQ8_KIND_CASE(int32_t);
    default: return DQ8_KIND_CASE(uint32_t);
  }
#undef DQ8_KIND_CASE
}
