// Running minimum / maximum of a float tensor, per tensor or per channel: the statistic
// the calibration observers of the quantization tool accumulate before they derive scales
// and zero points.  HBM-bound: 4 bytes read per element, a few bytes written per workgroup.
//
// Two passes, no atomics, so the result does not depend on the order workgroups finish in
// and a NaN anywhere in a channel's data makes that channel's minimum and maximum NaN:
//   1. every workgroup reduces a slab of the tensor to one (min, max) pair per channel it
//      touches and writes it to the workspace;
//   2. a small second kernel reduces each channel's pairs and folds them into the running
//      values the caller keeps.
// The tensor is viewed as [outer, channels, inner], row-major.
//  * inner > 1 (or one channel): "rows" of `inner` contiguous elements, row r belongs to
//    channel r % channels; a workgroup reduces one segment of up to 4096 elements of one row
//    (16 bytes per thread per load, four loads in flight), one sweep over the tensor by many
//    small workgroups, as in the quantize kernels;
//  * inner == 1 and more than one channel (channel = last axis): threads along the channels,
//    four channels each, a workgroup walks a block of rows.
#include <algorithm>
#include <limits>
#include <mutex>

#include "dq8_common.h"
#include "disc_q8.h"
#include "q8_elementwise.h"

#pragma clang fp contract(off)

namespace dq8 {
namespace {

constexpr int kThreads = 256;
constexpr int kSegment = 4096;   // elements of one row a workgroup reduces (row kernel)

struct MinMax {
  float lo, hi;
};

// min / max that keep a NaN once they have seen one
__device__ __forceinline__ void fold(MinMax& m, float v) {
  m.lo = v < m.lo ? v : m.lo;
  m.hi = v > m.hi ? v : m.hi;
  if (v != v) {
    m.lo = v;
    m.hi = v;
  }
}
__device__ __forceinline__ void fold(MinMax& m, const MinMax& o) {
  const bool nan = o.lo != o.lo || m.lo != m.lo;
  m.lo = o.lo < m.lo ? o.lo : m.lo;
  m.hi = o.hi > m.hi ? o.hi : m.hi;
  if (nan) {
    m.lo = std::numeric_limits<float>::quiet_NaN();
    m.hi = m.lo;
  }
}

__device__ __forceinline__ MinMax identity() {
  return {std::numeric_limits<float>::infinity(), -std::numeric_limits<float>::infinity()};
}

// all-lanes reduction inside a wave, then over the waves of the workgroup through LDS;
// the result is valid in thread 0
__device__ __forceinline__ MinMax block_reduce(MinMax m) {
  __shared__ MinMax part[kThreads / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    MinMax o;
    o.lo = __shfl_xor(m.lo, off, 64);
    o.hi = __shfl_xor(m.hi, off, 64);
    fold(m, o);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) part[wave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kThreads / 64; ++w) fold(m, part[w]);
  }
  return m;
}

// ---- pass 1, rows: workgroup b reduces piece b % segs of row b / segs; a piece is `chunks`
// consecutive segments of kSegment elements (one segment unless the row is so long that the
// number of pairs per channel would make the second pass noticeable)
template <bool VEC>
__global__ void __launch_bounds__(kThreads)
minmax_rows(const float* __restrict__ x, int64_t inner, int segs, int chunks,
            float2* __restrict__ partial) {
  const int64_t row = blockIdx.x / segs;
  const int seg = (int)(blockIdx.x - row * segs);
  const float* p = x + row * inner;
  MinMax m = identity();
  for (int ch = 0; ch < chunks; ++ch) {
    const int64_t begin = ((int64_t)seg * chunks + ch) * kSegment;
    if (begin >= inner) break;
    const int64_t end = begin + kSegment < inner ? begin + kSegment : inner;
    if (VEC) {
      // row starts are 16-byte aligned: inner % 4 == 0 and an aligned tensor
      const float4* p4 = reinterpret_cast<const float4*>(p);
      const int64_t b4 = begin / 4, e4 = end / 4;
      float4 v[4];
      bool have[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t i = b4 + threadIdx.x + (int64_t)u * kThreads;
        have[u] = i < e4;
        if (have[u]) v[u] = p4[i];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (have[u]) {
          fold(m, v[u].x);
          fold(m, v[u].y);
          fold(m, v[u].z);
          fold(m, v[u].w);
        }
    } else {
      for (int64_t i = begin + threadIdx.x; i < end; i += kThreads) fold(m, p[i]);
    }
  }
  m = block_reduce(m);
  if (threadIdx.x == 0) partial[blockIdx.x] = make_float2(m.lo, m.hi);
}

// ---- pass 1, channel = last axis: x [rows, nch]; thread (tx, ty) of block (bx, by) owns
// channels 4 * (bx * blockDim.x + tx) .. + 3 and walks rows by * rows_per_block + ty,
// + blockDim.y, ...; partial[by][channel]
template <bool VEC>
__global__ void __launch_bounds__(kThreads)
minmax_lastaxis(const float* __restrict__ x, int64_t rows, int nch, int rows_per_block,
                float2* __restrict__ partial) {
  __shared__ MinMax stage[kThreads][4];
  constexpr int W = VEC ? 4 : 1;
  const int c0 = (blockIdx.x * blockDim.x + threadIdx.x) * W;
  const int64_t r_begin = (int64_t)blockIdx.y * rows_per_block;
  const int64_t r_end = r_begin + rows_per_block < rows ? r_begin + rows_per_block : rows;
  MinMax m[4] = {identity(), identity(), identity(), identity()};
  if (c0 < nch) {
    const int64_t step = blockDim.y;
    int64_t r = r_begin + threadIdx.y;
    if (VEC) {
      // eight rows' loads in flight per thread
      for (; r + 7 * step < r_end; r += 8 * step) {
        float4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          v[u] = *reinterpret_cast<const float4*>(x + (r + u * step) * nch + c0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          fold(m[0], v[u].x);
          fold(m[1], v[u].y);
          fold(m[2], v[u].z);
          fold(m[3], v[u].w);
        }
      }
      for (; r < r_end; r += step) {
        const float4 v = *reinterpret_cast<const float4*>(x + r * nch + c0);
        fold(m[0], v.x);
        fold(m[1], v.y);
        fold(m[2], v.z);
        fold(m[3], v.w);
      }
    } else {
      for (; r < r_end; r += step) fold(m[0], x[r * nch + c0]);
    }
  }
  // rows handled by the threadIdx.y > 0 slices fold into slice 0 through LDS
  const int t = threadIdx.y * blockDim.x + threadIdx.x;
#pragma unroll
  for (int k = 0; k < W; ++k) stage[t][k] = m[k];
  __syncthreads();
  if (threadIdx.y == 0 && c0 < nch) {
    for (int y = 1; y < (int)blockDim.y; ++y)
#pragma unroll
      for (int k = 0; k < W; ++k) fold(m[k], stage[y * blockDim.x + threadIdx.x][k]);
#pragma unroll
    for (int k = 0; k < W; ++k)
      if (c0 + k < nch) partial[(int64_t)blockIdx.y * nch + c0 + k] = make_float2(m[k].lo, m[k].hi);
  }
}

// Scale and zero point of one channel from its running minimum and maximum, the observers'
// arithmetic (R tools/torch_quant/torch_quant/observer.py:134-163): separately rounded f32
// operations and true divisions.  `range` is (q_max - q_min) / 2 for the symmetric schemes and
// q_max - q_min for the affine ones.
struct QParamsOut {
  float* scale;         // null: only the minimum and maximum are wanted
  int32_t* zero_point;
  int32_t* status;      // 1: min <= max in every channel, 2: not so (host-visible memory)
  int symmetric;
  float range;
  int q_min, q_max;
};
__device__ __forceinline__ void qparams_of(const QParamsOut& q, float lo, float hi, float* scale, int* zero_point) {
  const float neg = lo < 0.0f ? lo : 0.0f, pos = hi > 0.0f ? hi : 0.0f;
  const float eps = std::numeric_limits<float>::epsilon();
  float s = (q.symmetric ? (-neg > pos ? -neg : pos) : pos - neg) / q.range;
  s = s > eps ? s : eps;
  int z = 0;
  if (!q.symmetric) {
    z = q.q_min - (int)rintf(neg / s);
    z = z < q.q_min ? q.q_min : (z > q.q_max ? q.q_max : z);
  }
  *scale = s;
  *zero_point = z;
}
__device__ __forceinline__ void qparams_one(const QParamsOut& q, int c, float lo, float hi) {
  float s;
  int z;
  qparams_of(q, lo, hi, &s, &z);
  q.scale[c] = s;
  q.zero_point[c] = z;
}
__device__ __forceinline__ void signal(int32_t* status, bool ok) {
  __hip_atomic_store(status, ok ? 1 : 2, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The same for many channels, behind pass 2: one workgroup, which also finds out whether every
// channel's minimum is at most its maximum (not so after a NaN).
__global__ void __launch_bounds__(1024)
minmax_qparams(const float* __restrict__ lo, const float* __restrict__ hi, int channels,
               const QParamsOut q) {
  bool ok = true;
  for (int c = threadIdx.x; c < channels; c += 1024) {
    const float a = lo[c], b = hi[c];
    ok = ok && a <= b;
    qparams_one(q, c, a, b);
  }
  const bool all = __syncthreads_and(ok);
  if (threadIdx.x == 0) signal(q.status, all);
}

// ---- pass 2, rows layout: one workgroup per channel c; its pairs are
// partial[(o * channels + c) * segs + s], o < outer, s < segs.  With a single channel the
// workgroup goes on to the channel's scale and zero point where they are wanted.
__global__ void __launch_bounds__(kThreads)
minmax_fold_rows(const float2* __restrict__ partial, int64_t outer, int channels, int segs,
                 float* __restrict__ min_io, float* __restrict__ max_io, const QParamsOut q) {
  const int c = blockIdx.x;
  MinMax m = identity();
  for (int64_t o = 0; o < outer; ++o) {
    const float2* row = partial + (o * channels + c) * segs;
    int s = threadIdx.x;
    for (; s + 3 * kThreads < segs; s += 4 * kThreads) {      // four loads in flight
      const float2 v0 = row[s], v1 = row[s + kThreads], v2 = row[s + 2 * kThreads],
                   v3 = row[s + 3 * kThreads];
      fold(m, MinMax{v0.x, v0.y});
      fold(m, MinMax{v1.x, v1.y});
      fold(m, MinMax{v2.x, v2.y});
      fold(m, MinMax{v3.x, v3.y});
    }
    for (; s < segs; s += kThreads) {
      const float2 v = row[s];
      fold(m, MinMax{v.x, v.y});
    }
  }
  m = block_reduce(m);
  if (threadIdx.x == 0) {
    fold(m, MinMax{min_io[c], max_io[c]});
    min_io[c] = m.lo;
    max_io[c] = m.hi;
    if (q.scale) {
      qparams_one(q, c, m.lo, m.hi);
      signal(q.status, m.lo <= m.hi);
    }
  }
}

// ---- pass 2, rows layout with few pairs per channel: one thread per channel
__global__ void __launch_bounds__(kThreads)
minmax_fold_rows_small(const float2* __restrict__ partial, int64_t outer, int channels, int segs,
                       float* __restrict__ min_io, float* __restrict__ max_io) {
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= channels) return;
  MinMax m = identity();
  for (int64_t o = 0; o < outer; ++o)
    for (int s = 0; s < segs; ++s) {
      const float2 v = partial[(o * channels + c) * segs + s];
      fold(m, MinMax{v.x, v.y});
    }
  fold(m, MinMax{min_io[c], max_io[c]});
  min_io[c] = m.lo;
  max_io[c] = m.hi;
}

// ---- pass 2, last-axis layout: pairs partial[g * channels + c].  A workgroup takes 64
// channels; its four waves each reduce every fourth group and meet in LDS.
__global__ void __launch_bounds__(kThreads)
minmax_fold_lastaxis(const float2* __restrict__ partial, int groups, int channels,
                     float* __restrict__ min_io, float* __restrict__ max_io) {
  __shared__ MinMax part[kThreads];
  const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  MinMax m = identity();
  if (c < channels) {
    for (int g = slice; g < groups; g += kThreads / 64) {
      const float2 v = partial[(int64_t)g * channels + c];
      fold(m, MinMax{v.x, v.y});
    }
  }
  part[threadIdx.x] = m;
  __syncthreads();
  if (slice == 0 && c < channels) {
#pragma unroll
    for (int w = 1; w < kThreads / 64; ++w) fold(m, part[w * 64 + lane]);
    fold(m, MinMax{min_io[c], max_io[c]});
    min_io[c] = m.lo;
    max_io[c] = m.hi;
  }
}

// ---- pass 2 and the fake quantization in one launch.  Every workgroup (per tensor) or wave (per
// row) folds the pairs and the running values it needs itself, instead of waiting for a kernel that
// does so once: at calibration sizes a step is launches and trips to memory, and the pairs come from
// the L2 (a step in a loop, per row, 740 x 240 21.1 -> 17.5 us, 71 x 1328 20.7 -> 16.4; per tensor, where
// one launch is saved and not two, 3072 x 768 18.2 -> 17.0).
// Workgroup 0 also stores the running values, scale and zero point and gives the answer.  Others may
// read a running value before or after it is stored: folding the same pairs into the result again
// gives the result, bit for bit.
struct FakeRange {
  float s, y, lo, hi;
  int z;
  bool fast;
  __device__ __forceinline__ FakeRange(const QParamsOut& q, const MinMax& m) {
    qparams_of(q, m.lo, m.hi, &s, &z);
    y = 1.0f / s;
    fast = elementwise::divisor_in_fast_range(s);
    lo = (float)q.q_min;
    hi = (float)q.q_max;
  }
  __device__ __forceinline__ float4 operator()(const float4& v) const {
    using namespace elementwise;
    return fast ? fake4_by_constant<1>(v, s, y, z, lo, hi)
                : make_float4(fake_one<1>(v.x, s, z, lo, hi), fake_one<1>(v.y, s, z, lo, hi),
                              fake_one<1>(v.z, s, z, lo, hi), fake_one<1>(v.w, s, z, lo, hi));
  }
};

// per tensor: n4 groups of four in tiles of 1024, `tiles` of them dealt over the workgroups
__global__ void __launch_bounds__(kThreads)
fold_fake_quant_tensor(const float4* __restrict__ x, float4* __restrict__ out, int64_t n4, int tiles,
                       const float2* __restrict__ partial, int segs, float* min_io, float* max_io,
                       const QParamsOut q) {
  __shared__ MinMax all;
  float4 v[4];
  auto load = [&](int t) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t i = (int64_t)t * 1024 + u * kThreads + threadIdx.x;
      v[u] = x[i < n4 ? i : n4 - 1];
    }
  };
  load(blockIdx.x);                        // (the data on its way under the pairs)
  MinMax m = identity();
  for (int s0 = threadIdx.x; s0 < segs; s0 += 4 * kThreads) {
    float2 pr[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) pr[u] = partial[s0 + u * kThreads < segs ? s0 + u * kThreads : s0];
#pragma unroll
    for (int u = 0; u < 4; ++u) fold(m, MinMax{pr[u].x, pr[u].y});
  }
  m = block_reduce(m);
  if (threadIdx.x == 0) {
    fold(m, MinMax{min_io[0], max_io[0]});
    all = m;
  }
  __syncthreads();
  m = all;
  const FakeRange f(q, m);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    min_io[0] = m.lo;
    max_io[0] = m.hi;
    q.scale[0] = f.s;
    q.zero_point[0] = f.z;
    signal(q.status, m.lo <= m.hi);
  }
  for (int t = blockIdx.x;;) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t i = (int64_t)t * 1024 + u * kThreads + threadIdx.x;
      if (i < n4) dq8::st_stream(&out[i], f(v[u]));
    }
    t += gridDim.x;
    if (t >= tiles) break;
    load(t);
  }
}

// per row (channel = row): a wave per piece of 256 groups of four of a row; workgroup 0 stores the
// channels' results instead
__device__ __forceinline__ MinMax row_range(const float2* __restrict__ partial, int segs, int first, int step,
                                            int64_t row, const float* min_io, const float* max_io) {
  const MinMax state = {min_io[row], max_io[row]};
  MinMax m = identity();
  for (int s = first; s < segs; s += step) {
    const float2 pr = partial[row * segs + s];
    fold(m, MinMax{pr.x, pr.y});
  }
  for (int off = step >> 1; off > 0; off >>= 1) {
    MinMax o;
    o.lo = __shfl_xor(m.lo, off, 64);
    o.hi = __shfl_xor(m.hi, off, 64);
    fold(m, o);
  }
  fold(m, state);
  return m;
}

__global__ void __launch_bounds__(kThreads)
fold_fake_quant_rows(const float4* __restrict__ x, float4* __restrict__ out, int rows, int inner4, int pieces,
                     const float2* __restrict__ partial, int segs, float* min_io, float* max_io,
                     const QParamsOut q) {
  if (blockIdx.x == 0) {
    bool ok = true;
#pragma unroll 4
    for (int c = threadIdx.x; c < rows; c += kThreads) {
      const MinMax m = row_range(partial, segs, 0, 1, c, min_io, max_io);
      ok = ok && m.lo <= m.hi;
      min_io[c] = m.lo;
      max_io[c] = m.hi;
      qparams_one(q, c, m.lo, m.hi);
    }
    const bool every = __syncthreads_and(ok);
    if (threadIdx.x == 0) signal(q.status, every);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int64_t unit = (int64_t)(blockIdx.x - 1) * 4 + (threadIdx.x >> 6);
  const int64_t row = unit / pieces;
  if (row >= rows) return;
  const int first = (int)(unit - row * pieces) * 256;
  const float4* px = x + row * inner4;
  float4 v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = first + u * 64 + lane;
    v[u] = px[i < inner4 ? i : inner4 - 1];
  }
  // (one pair a row: every lane reads it)
  const MinMax m = segs == 1 ? row_range(partial, 1, 0, 1, row, min_io, max_io)
                             : row_range(partial, segs, lane, 64, row, min_io, max_io);
  const FakeRange f(q, m);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = first + u * 64 + lane;
    if (i < inner4) dq8::st_stream(&out[row * inner4 + i], f(v[u]));
  }
}

struct Plan {
  bool last_axis;
  int segs;             // rows layout: pieces per row
  int chunks;           // rows layout: segments per piece
  int64_t blocks;       // rows layout: workgroups of pass 1
  int bx, by, gx, gy, rows_per_block;   // last-axis layout
  int64_t pairs;        // (min, max) pairs in the workspace
};

bool make_plan(int64_t outer, int64_t channels, int64_t inner, bool vec, Plan* p) {
  *p = Plan{};
  if (inner == 1 && channels > 1) {
    p->last_axis = true;
    const int64_t units = vec ? channels / 4 : channels;
    int bx = 1;
    while (bx < kThreads && bx < units) bx *= 2;
    p->bx = bx;
    p->by = kThreads / bx;
    p->gx = (int)ceil_div(units, bx);
    // Row blocks: about 512 workgroups in all for the four-channels-per-thread form (eight
    // 16-byte loads in flight per thread), at least 64 rows each.  The same split is used for the one-channel-per-thread form, so
    // that the workspace does not depend on the alignment of the tensor.
    const int64_t units4 = ceil_div(channels, 4);
    const int64_t gx4 = ceil_div(units4, std::min<int64_t>(kThreads, units4));
    const int64_t gy_target = std::max<int64_t>(1, 512 / gx4);
    const int64_t rpb = std::max<int64_t>(ceil_div(outer, gy_target), 64);
    const int64_t gy = ceil_div(outer, rpb);
    if (gy > 65535 || rpb > (1 << 30)) return false;
    p->gy = (int)gy;
    p->rows_per_block = (int)rpb;
    p->pairs = gy * channels;
    return true;
  }
  const int64_t rows = outer * channels;
  // at most about 8192 pairs per channel, at most 64 segments per workgroup
  const int64_t all = ceil_div(inner, kSegment);
  const int64_t chunks = std::min<int64_t>(64, std::max<int64_t>(1, ceil_div(all * outer, 8192)));
  const int64_t segs = ceil_div(all, chunks);
  if (segs > (1 << 30) || rows * segs >= (1LL << 31)) return false;
  p->segs = (int)segs;
  p->chunks = (int)chunks;
  p->blocks = rows * segs;
  p->pairs = p->blocks;
  return true;
}

// Whether the fake quantization folds the pairs itself, one launch behind pass 1: while what is folded
// more than once, or by workgroup 0 on a thread a row, stays small.  A step in a loop, in one launch /
// with a kernel that folds once:
//  * a tensor, up to 4096 pairs folded by at most 1024 workgroups (32 MB from the L2s): 3 M elements 16.1 /
//    16.4 us, 8 M 20.5 / 22.8, 16 M 37.5 / 38.5;
//  * rows of up to six pairs, fewer than 1024 rows (from there on the other form folds a thread a row as
//    well) and 8 M elements: 64 x 24576 14.7 / 16.8, 512 x 4096 15.4 / 17.0, 740 x 8192 21.0 / 21.6; beyond,
//    2 x 1048576 39 / 18, 64 x 131072 28.5 / 25.0, 1024 x 3072 17.2 / 17.0, 2048 x 1024 17.9 / 16.7.
bool fold_plan(int64_t outer, int64_t channels, int64_t inner, Plan* p) {
  if (outer != 1 || inner % 4 != 0 || !make_plan(1, channels, inner, true, p)) return false;
  return channels == 1 ? p->segs <= 4096 : channels < 1024 && p->segs <= 6 && channels * inner <= (1 << 23);
}

}  // namespace

bool observe_folds_range(int64_t outer, int64_t channels, int64_t inner) {
  Plan p;
  return fold_plan(outer, channels, inner, &p);
}

}  // namespace dq8

using namespace dq8;

extern "C" size_t dq8_minmax_workspace_bytes(int64_t outer, int64_t channels, int64_t inner) {
  if (outer <= 0 || channels <= 0 || inner <= 0) return 0;
  Plan p;
  // (the space needed does not depend on whether the vectorised kernels can be used)
  if (!make_plan(outer, channels, inner, false, &p)) return 0;
  return (size_t)p.pairs * sizeof(float2);
}

namespace {

// Shared by the entry points: both passes with the (min, max) pairs in `partial`.  Pass 1
// writes every pair pass 2 reads, so the scratch needs no particular contents beforehand.
// `q`: of a single channel (null where scale and zero point are not wanted).
int run_minmax(const float* x, int64_t outer, int64_t channels, int64_t inner,
               float* min_io, float* max_io, float2* partial, const Plan& p, bool vec,
               hipStream_t st, const QParamsOut* q = nullptr) {
  if (p.last_axis) {
    const dim3 grid((unsigned)p.gx, (unsigned)p.gy), block((unsigned)p.bx, (unsigned)p.by);
    if (vec)
      hipLaunchKernelGGL(minmax_lastaxis<true>, grid, block, 0, st, x, outer, (int)channels,
                         p.rows_per_block, partial);
    else
      hipLaunchKernelGGL(minmax_lastaxis<false>, grid, block, 0, st, x, outer, (int)channels,
                         p.rows_per_block, partial);
    if (int s = check_hip(hipGetLastError(), "minmax_lastaxis launch")) return s;
    hipLaunchKernelGGL(minmax_fold_lastaxis, dim3((unsigned)ceil_div(channels, 64)),
                       dim3(kThreads), 0, st, partial, p.gy, (int)channels, min_io, max_io);
    return check_hip(hipGetLastError(), "minmax_fold_lastaxis launch");
  }
  if (vec)
    hipLaunchKernelGGL(minmax_rows<true>, dim3((unsigned)p.blocks), dim3(kThreads), 0, st, x,
                       inner, p.segs, p.chunks, partial);
  else
    hipLaunchKernelGGL(minmax_rows<false>, dim3((unsigned)p.blocks), dim3(kThreads), 0, st, x,
                       inner, p.segs, p.chunks, partial);
  if (int s = check_hip(hipGetLastError(), "minmax_rows launch")) return s;
  if (outer * p.segs <= 32 && channels >= 1024)
    hipLaunchKernelGGL(minmax_fold_rows_small, dim3((unsigned)ceil_div(channels, kThreads)),
                       dim3(kThreads), 0, st, partial, outer, (int)channels, p.segs, min_io, max_io);
  else
    hipLaunchKernelGGL(minmax_fold_rows, dim3((unsigned)channels), dim3(kThreads), 0, st, partial,
                       outer, (int)channels, p.segs, min_io, max_io, q ? *q : QParamsOut{});
  return check_hip(hipGetLastError(), "minmax_fold_rows launch");
}

}  // namespace

extern "C" int dq8_minmax(const float* x, int64_t outer, int64_t channels, int64_t inner,
                          float* min_io, float* max_io, void* workspace,
                          size_t workspace_bytes, void* stream) {
  clear_error();
  DQ8_REQUIRE(outer >= 0 && channels >= 0 && inner >= 0, "dq8_minmax: negative extent");
  if (outer == 0 || channels == 0 || inner == 0) return 0;   // nothing observed: state kept
  DQ8_REQUIRE(x && min_io && max_io, "dq8_minmax: null pointer");
  DQ8_REQUIRE(channels < (1LL << 31), "dq8_minmax: too many channels");
  const bool last_axis = inner == 1 && channels > 1;
  const bool vec = aligned(x, 16) && (last_axis ? channels % 4 == 0 : inner % 4 == 0);
  Plan p;
  DQ8_REQUIRE(make_plan(outer, channels, inner, vec, &p), "dq8_minmax: tensor too large");
  DQ8_REQUIRE(workspace && workspace_bytes >= (size_t)p.pairs * sizeof(float2),
              "dq8_minmax: workspace too small (see dq8_minmax_workspace_bytes)");
  return run_minmax(x, outer, channels, inner, min_io, max_io,
                    static_cast<float2*>(workspace), p, vec, (hipStream_t)stream);
}

// A whole observation step: the running minimum and maximum, then scale and zero point from
// them, with nothing read back in between.
extern "C" int dq8_observe(const float* x, int64_t outer, int64_t channels, int64_t inner,
                           float* min_io, float* max_io, int symmetric, int32_t q_min,
                           int32_t q_max, float* scale, int32_t* zero_point, int32_t* status,
                           void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  DQ8_REQUIRE(outer > 0 && channels > 0 && inner > 0, "dq8_observe: empty tensor");
  DQ8_REQUIRE(x && min_io && max_io && scale && zero_point && status, "dq8_observe: null pointer");
  DQ8_REQUIRE(channels < (1LL << 31), "dq8_observe: too many channels");
  DQ8_REQUIRE(q_min < q_max && q_min >= -32768 && q_max <= 65535,
              "dq8_observe: quant_min/quant_max outside the 8- and 16-bit ranges");
  const bool last_axis = inner == 1 && channels > 1;
  const bool vec = aligned(x, 16) && (last_axis ? channels % 4 == 0 : inner % 4 == 0);
  Plan p;
  DQ8_REQUIRE(make_plan(outer, channels, inner, vec, &p), "dq8_observe: tensor too large");
  DQ8_REQUIRE(workspace && workspace_bytes >= (size_t)p.pairs * sizeof(float2),
              "dq8_observe: workspace too small (see dq8_minmax_workspace_bytes)");
  const float full = (float)(q_max - q_min);
  const QParamsOut q = {scale, zero_point, status, symmetric, symmetric ? full / 2 : full, q_min, q_max};
  if (int s = run_minmax(x, outer, channels, inner, min_io, max_io, static_cast<float2*>(workspace),
                         p, vec, (hipStream_t)stream, channels == 1 ? &q : nullptr))
    return s;
  if (channels == 1) return 0;
  hipLaunchKernelGGL(minmax_qparams, dim3(1), dim3(1024), 0, (hipStream_t)stream, min_io, max_io,
                     (int)channels, q);
  return check_hip(hipGetLastError(), "minmax_qparams launch");
}

// The observation step and the fake quantization of the same tensor with its result.
extern "C" int dq8_observe_fake_quant(const float* x, float* out, int64_t outer, int64_t channels, int64_t inner,
                                      float* min_io, float* max_io, int symmetric, int32_t q_min, int32_t q_max,
                                      float* scale, int32_t* zero_point, int32_t* status, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  clear_error();
  DQ8_REQUIRE(outer > 0 && channels > 0 && inner > 0, "dq8_observe_fake_quant: empty tensor");
  DQ8_REQUIRE(x && out && min_io && max_io && scale && zero_point && status,
              "dq8_observe_fake_quant: null pointer");
  DQ8_REQUIRE(channels < (1LL << 31), "dq8_observe_fake_quant: too many channels");
  DQ8_REQUIRE(q_min < q_max && q_min >= -32768 && q_max <= 65535,
              "dq8_observe_fake_quant: quant_min/quant_max outside the 8- and 16-bit ranges");
  Plan p;
  if (aligned(x, 16) && aligned(out, 16) && fold_plan(outer, channels, inner, &p)) {
    DQ8_REQUIRE(workspace && workspace_bytes >= (size_t)p.pairs * sizeof(float2),
                "dq8_observe_fake_quant: workspace too small (see dq8_minmax_workspace_bytes)");
    hipStream_t st = (hipStream_t)stream;
    float2* partial = static_cast<float2*>(workspace);
    const float full = (float)(q_max - q_min);
    const QParamsOut q = {scale, zero_point, status, symmetric, symmetric ? full / 2 : full, q_min, q_max};
    hipLaunchKernelGGL(minmax_rows<true>, dim3((unsigned)p.blocks), dim3(kThreads), 0, st, x, inner, p.segs,
                       p.chunks, partial);
    if (int s = check_hip(hipGetLastError(), "minmax_rows launch")) return s;
    if (channels == 1) {
      const int64_t tiles = ceil_div(inner / 4, 1024);
      hipLaunchKernelGGL(fold_fake_quant_tensor, dim3((unsigned)std::min<int64_t>(tiles, 1024)), dim3(kThreads), 0,
                         st, reinterpret_cast<const float4*>(x), reinterpret_cast<float4*>(out), inner / 4,
                         (int)tiles, partial, p.segs, min_io, max_io, q);
    } else {
      const int64_t pieces = ceil_div(inner / 4, 256);
      hipLaunchKernelGGL(fold_fake_quant_rows, dim3((unsigned)(1 + ceil_div(channels * pieces, 4))), dim3(kThreads),
                         0, st, reinterpret_cast<const float4*>(x), reinterpret_cast<float4*>(out), (int)channels,
                         (int)(inner / 4), (int)pieces, partial, p.segs, min_io, max_io, q);
    }
    return check_hip(hipGetLastError(), "fold_fake_quant launch");
  }
  if (int s = dq8_observe(x, outer, channels, inner, min_io, max_io, symmetric, q_min, q_max, scale, zero_point,
                          status, workspace, workspace_bytes, stream))
    return s;
  return dq8_fake_quant(x, out, outer, channels, inner, scale, zero_point, channels, q_min, q_max,
                        DQ8_ROUND_HALF_TO_EVEN, stream);
}

// ---- the same with the pairs in memory the library brings along -------------------------
// For callers that cannot allocate (code under graph capture, serving loops that forbid
// hipMalloc): the (min, max) pairs of pass 1 live in a fixed array in device memory.  Every
// device the library runs on holds its own copy of the array at its own address, looked up
// once per device, with that device current, and kept; host code never uses the array's
// name for anything else.
namespace {

constexpr size_t kStaticScratchBytes = 4u << 20;   // 524288 (min, max) pairs
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// device address of `scratch` on the current device (nullptr + error status on failure)
int static_scratch(void** out) {
  int dev = 0;
  if (int s = check_hip(hipGetDevice(&dev), "hipGetDevice")) return s;
  DQ8_REQUIRE(dev >= 0 && dev < kMaxDevices, "dq8_minmax_static: device ordinal out of range");
  std::lock_guard<std::mutex> guard(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (int s = check_hip(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)),
                          "hipGetSymbolAddress(scratch)"))
      return s;
    DQ8_REQUIRE(ptr != nullptr, "dq8_minmax_static: no device address for the scratch array");
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

}  // namespace

extern "C" size_t dq8_minmax_static_max_bytes(void) { return kStaticScratchBytes; }

extern "C" int dq8_minmax_static(const float* x, int64_t outer, int64_t channels, int64_t inner,
                                 float* min_io, float* max_io, void* stream) {
  clear_error();
  DQ8_REQUIRE(outer >= 0 && channels >= 0 && inner >= 0, "dq8_minmax_static: negative extent");
  if (outer == 0 || channels == 0 || inner == 0) return 0;
  DQ8_REQUIRE(x && min_io && max_io, "dq8_minmax_static: null pointer");
  DQ8_REQUIRE(channels < (1LL << 31), "dq8_minmax_static: too many channels");
  const bool last_axis = inner == 1 && channels > 1;
  const bool vec = aligned(x, 16) && (last_axis ? channels % 4 == 0 : inner % 4 == 0);
  Plan p;
  DQ8_REQUIRE(make_plan(outer, channels, inner, vec, &p), "dq8_minmax_static: tensor too large");
  DQ8_REQUIRE((size_t)p.pairs * sizeof(float2) <= kStaticScratchBytes,
              "dq8_minmax_static: this tensor needs " +
                  std::to_string((size_t)p.pairs * sizeof(float2)) +
                  " bytes of scratch, more than the built-in " +
                  std::to_string(kStaticScratchBytes) + "; use dq8_minmax with a workspace");
  void* ptr = nullptr;
  if (int s = static_scratch(&ptr)) return s;
  return run_minmax(x, outer, channels, inner, min_io, max_io,
                    static_cast<float2*>(ptr), p, vec, (hipStream_t)stream);
}
