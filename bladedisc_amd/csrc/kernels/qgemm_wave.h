// int8 MFMA GEMM / implicit-GEMM convolution for launches with a tile or two to a compute unit: the k tiles
// of an output tile are dealt out over the waves of its workgroup, and no wave waits for another before
// the sums meet.
//
// What bounds such a launch is the CU's load path.  Direct-to-LDS loads of 8 rows x 128 B out of the L2 run at
// 60 B a clock and CU as long as some wave always has the next one to issue.  Waves that share a tile, a barrier
// per k tile, issue in step and wait in step, and the path idles in between: the operand loads alone of 192
// tiles of 64 x 64 over 3072 of k (393 KB a CU) take 4.5 us with a barrier per k tile on four waves, 3.6 on
// eight, whatever the number of stages (2 .. 8), and 2.6 us without one.  Hence:
//  * every wave multiplies the whole BM x BN tile, over k tiles w, w + NW, w + 2 NW ... of 128, out of
//    LDS stages that only it loads and reads: its s_waitcnt is all the synchronisation there is;
//  * a wave holds all fragments of a k tile in registers before it refills the stage, loads and matrix
//    instructions in turn;
//  * the NW partial tiles are added through LDS at the end, each wave collecting the fragments that it
//    then runs the epilogue on (a 64 x 64 tile on four waves: one each).
// LDS: 1 KiB blocks of 8 rows x 128 B as in qgemm_pipelined.h, chunk c of row r in slot c ^ r; blocks lie 1152
// bytes apart, which puts rows r and r + 8 of a fragment into different halves of the banks and leaves
// every lane with the same chunk in every block it loads.
// Requires what the pipelined kernel does: K % 16 == 0, 16-byte aligned, k-contiguous operands, 32-bit
// offsets.  ROWMAP, ZP, WORDS (rows on four bytes): see qgemm_pipelined.h.
#ifndef DQ8_QGEMM_WAVE_H_
#define DQ8_QGEMM_WAVE_H_

#include "lds_direct.h"
#include "qgemm_device.h"

namespace dq8 {

constexpr int kWaveBlock = 1152;   // bytes between two blocks of 8 rows
constexpr int qgemm_wave_lds(int fm, int fn, int nw, int stages) { return nw * stages * (fm + fn) * 4 * kWaveBlock; }

template <int FM, int FN, int NW, int STAGES, bool CONV, int EPI, bool ROWMAP = false, bool ZP = false, bool WORDS = false>
__global__ void __launch_bounds__(NW * 64) qgemm_wave_kernel(const MainParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BK = 128, NKS = BK / 32;
  constexpr int BM = FM * 32, BN = FN * 32, NT = NW * 64;
  constexpr int A_LD = BM / 8, B_LD = BN / 8, LD = A_LD + B_LD;
  constexpr int STAGE = LD * kWaveBlock;
  static_assert((STAGES - 1) * LD <= 63, "vmcnt is a 6-bit counter");
  // what a wave takes to the epilogue: a fragment, or a row of two where the fragments outnumber the waves
  constexpr int ON = FM * FN > NW ? 2 : 1;
  constexpr int OWNERS = FM * FN / ON;
  static_assert(OWNERS <= NW && FN % ON == 0, "every fragment has an owner");

  extern __shared__ __attribute__((aligned(1024))) int8_t smem_all[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int8_t* smem = smem_all + wave * (STAGES * STAGE);

  int tm, tn;
  tile_coords(blockIdx.x, gridDim.x, p.tiles_m, p.tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int KT = (p.K + BK - 1) / BK;
  const int nt = (KT - wave + NW - 1) / NW;          // k tiles of this wave (may be none)

  constexpr int64_t kMaxRecords = 0x7fffffff;
  constexpr int kOutOfRange = (int)0x80000000;
  static_assert(!(CONV && ROWMAP), "rows mapped to pixels: a form of the plain GEMM");
  const int8_t* a_base = CONV || ROWMAP ? p.A : p.A + (int64_t)m0 * p.lda;
  const int64_t a_valid = CONV || ROWMAP ? p.conv_bytes : (int64_t)(p.M - m0 - 1) * p.lda + p.K;
  const int64_t w_valid = (int64_t)(p.N - n0 - 1) * p.ldw + p.K;
  const v4i a_rsrc = make_rsrc(a_base, a_valid < kMaxRecords ? a_valid : kMaxRecords);
  const v4i w_rsrc = make_rsrc(p.W + (int64_t)n0 * p.ldw, w_valid < kMaxRecords ? w_valid : kMaxRecords);
  const unsigned lds_base = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(size_t)(lds_void_t*)smem);

  // ahead of the loads that are counted below
  EarlyColRaw<EPI, NT, BN> early;
  early.request(p.epi, n0);

  // load i of a k tile: rows 8 i .. 8 i + 7, lane -> row lane / 8, slot lane % 8, chunk slot ^ row
  const int lr = lane >> 3;
  const int kc = ((lane & 7) ^ lr) << 4;
  int a_off[A_LD];
  // conv: the row's first input pixel (coordinates, and byte offset of its channel 0)
  int a_h[CONV ? A_LD : 1], a_w[CONV ? A_LD : 1];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) {
    if (CONV || ROWMAP) {
      const int m = ROWMAP ? min(m0 + i * 8 + lr, p.M - 1) : m0 + i * 8 + lr;
      const int hw = p.Ho * p.Wo;
      const int n_img = m / hw, rem = m - n_img * hw;
      const int ho = rem / p.Wo, wo = rem - ho * p.Wo;
      if (CONV) {
        // rows past M get a coordinate no tap can bring back into the image
        a_h[CONV ? i : 0] = m < p.M ? ho * p.sh - p.pad_t : -(1 << 24);
        a_w[CONV ? i : 0] = wo * p.sw_ - p.pad_l;
        a_off[i] = m < p.M ? ((n_img * p.H + ho * p.sh - p.pad_t) * p.Wd + a_w[CONV ? i : 0]) * p.Ci : 0;
      } else {
        a_off[i] = ((n_img * p.H + ho * p.sh) * p.Wd + wo * p.sw_) * p.Ci + kc;
      }
    } else {
      a_off[i] = (i * 8 + lr) * (int)p.lda + kc;
    }
  }
  const int b_off0 = lr * (int)p.ldw + kc;
  const int b_step = 8 * (int)p.ldw;

  // The k tile whose loads are issued next: inside K, and (conv) the tap of the lane's chunk, advanced by NW
  // tiles per call.
  int k_next = wave * BK;
  int t_koff = kOutOfRange, t_dh = 0, t_dw = 0, t_off = 0;
  int c_ci = 0, c_kh = 0, c_kw = 0, d_ci = 0, d_kh = 0, d_kw = 0;
  if (CONV) {
    const unsigned k = (unsigned)(k_next + kc);
    const unsigned tap = k / (unsigned)p.Ci;
    c_ci = (int)(k - tap * (unsigned)p.Ci);
    c_kh = (int)(tap / (unsigned)p.Kw);
    c_kw = (int)(tap - (unsigned)c_kh * (unsigned)p.Kw);
    const int d_tap = NW * BK / p.Ci;
    d_ci = NW * BK - d_tap * p.Ci;
    d_kh = d_tap / p.Kw;
    d_kw = d_tap - d_kh * p.Kw;
  }
  auto tile_setup = [&]() {
    t_koff = k_next + kc < p.K ? k_next - (WORDS ? max(k_next + kc + 16 - p.K, 0) : 0) : kOutOfRange;
    k_next += NW * BK;
    if (CONV) {
      t_dh = c_kh * p.dh;
      t_dw = c_kw * p.dw;
      t_off = (t_dh * p.Wd + t_dw) * p.Ci + c_ci;
      c_ci += d_ci;
      const bool carry = c_ci >= p.Ci;
      c_ci -= carry ? p.Ci : 0;
      c_kw += d_kw + (carry ? 1 : 0);                  // (< 2 Kw)
      const bool wrap = c_kw >= p.Kw;
      c_kw -= wrap ? p.Kw : 0;
      c_kh += d_kh + (wrap ? 1 : 0);
    }
  };
  auto issue_load = [&](int i, unsigned at) {          // (i: a constant once unrolled)
    if (i < A_LD) {
      int voff = a_off[i < A_LD ? i : 0] + t_koff;     // (2^31 and a row's offset: past every descriptor)
      if (CONV) {
        const int hi = a_h[CONV && i < A_LD ? i : 0] + t_dh, wi = a_w[CONV && i < A_LD ? i : 0] + t_dw;
        const bool ok = t_koff != kOutOfRange && (unsigned)hi < (unsigned)p.H && (unsigned)wi < (unsigned)p.Wd;
        voff = ok ? a_off[i < A_LD ? i : 0] + t_off : kOutOfRange;
      }
      buffer_load_lds_b128(a_rsrc, at + i * kWaveBlock, voff);
    } else {
      buffer_load_lds_b128(w_rsrc, at + i * kWaveBlock, b_off0 + (i - A_LD) * b_step + t_koff);
    }
  };

  // fragment i of an operand: blocks 4 i .. 4 i + 3, row lane % 32, k-chunk 2 ks + lane / 32
  int frag_off[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    frag_off[ks] = ((lane >> 3) & 3) * kWaveBlock + (lane & 7) * 128 + (((2 * ks + (lane >> 5)) ^ (lane & 7)) << 4);

  v16i acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;
  int w_sum[ZP ? FN : 1];            // of the weights this wave has multiplied: row lane % 32, its half of k
#pragma unroll
  for (int j = 0; j < (ZP ? FN : 1); ++j) w_sum[j] = 0;

#pragma unroll
  for (int t = 0; t < STAGES; ++t)
    if (t < nt) {
      tile_setup();
#pragma unroll
      for (int i = 0; i < LD; ++i) issue_load(i, lds_base + t * STAGE);
    }

  // WORDS: whether the end of the rows is in this wave's last tile
  const bool row_end = WORDS && (p.K & 15) != 0 && nt > 0 && wave + (nt - 1) * NW == KT - 1;

  // MORE: tile t + STAGES exists and is loaded; else at most `behind` tiles are on their way behind tile t
  auto k_tile = [&](auto more_c, int st, bool last) {
    constexpr bool more = decltype(more_c)::value != 0;
    const int8_t* base = smem + st * STAGE;
    v4i fa[NKS][FM], fb[NKS][FN];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[ks][i] = *(const v4i*)(base + i * 4 * kWaveBlock + frag_off[ks]);
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[ks][j] = *(const v4i*)(base + (FM + j) * 4 * kWaveBlock + frag_off[ks]);
    }
    if (more) {
      tile_setup();
      // the stage is this wave's alone: free once its fragments are in registers
      __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(63));
      __builtin_amdgcn_sched_barrier(0);
    }
    if (WORDS && !more && last && row_end) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        if (ks == (p.K & (BK - 1)) / 32)
#pragma unroll
          for (int j = 0; j < FN; ++j) clear_row_end(fb[ks][j], p.K, lane);
    }
    constexpr int MF = NKS * FM * FN;
    static_for<MF>([&](auto mc) {
      constexpr int x = decltype(mc)::value, ks = x / (FM * FN), i = x / FN % FM, j = x % FN;
      if constexpr (more) {
#pragma unroll
        for (int l = x * LD / MF; l < (x + 1) * LD / MF; ++l) issue_load(l, lds_base + st * STAGE);
      }
      if constexpr (ZP && i == 0) {
#pragma unroll
        for (int c = 0; c < 4; ++c) w_sum[j] = __builtin_amdgcn_sdot4(fb[ks][j][c], 0x01010101, w_sum[j], false);
      }
      acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[ks][j], fa[ks][i], acc[i][j], 0, 0, 0);
      if (more) __builtin_amdgcn_sched_barrier(0);
    });
  };
  int t = 0, st = 0;
  for (; t + STAGES < nt; ++t) {
    // (tile t: older than the STAGES - 1 behind it)
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((STAGES - 1) * LD));
    asm volatile("" ::: "memory");
    k_tile(IntC<1>(), st, false);
    st = st + 1 == STAGES ? 0 : st + 1;
  }
  for (; t < nt; ++t) {
    static_for<STAGES>([&](auto ac) {
      constexpr int a = decltype(ac)::value;
      if (a == nt - t - 1) __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(a * LD));
    });
    asm volatile("" ::: "memory");
    k_tile(IntC<0>(), st, t == nt - 1);
    st = st + 1 == STAGES ? 0 : st + 1;
  }
  ColParams col[EarlyColRaw<EPI, NT, BN>::kPerThread];
  early.finish(p.epi, col);

  if constexpr (ZP) {
    // -zx times the sums, from a lane per channel to the accumulators' layout, through the wave's own LDS
    int* mine = reinterpret_cast<int*>(smem);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int s = w_sum[j] + __shfl_xor(w_sum[j], 32, 64);
      mine[j * 32 + (lane & 31)] = (int)(0u - (unsigned)p.zx * (unsigned)s);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v4i c = *reinterpret_cast<const v4i*>(&mine[j * 32 + 8 * g + 4 * (lane >> 5)]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < FM; ++i) acc[i][j][4 * g + q] += c[q];
      }
  }

  // ---- the waves' sums: fragment f to its owner f / ON, 16 bytes a lane
  __syncthreads();                                     // every wave is done with its stages
  const bool owner = OWNERS == NW || wave < OWNERS;
  // parked: for every fragment NW - 1 partial ones (those of the waves in turn, the owner's left out)
  auto slot = [&](int f, int w) {
    const int own = f / ON;
    return reinterpret_cast<v4i*>(smem_all) + (f * (NW - 1) + (w > own ? w - 1 : w)) * 256 + lane;
  };
#pragma unroll
  for (int f = 0; f < FM * FN; ++f)
    if (f / ON != wave) {
      v4i* dst = slot(f, wave);
#pragma unroll
      for (int g = 0; g < 4; ++g)
        dst[g * 64] = (v4i){acc[f / FN][f % FN][4 * g], acc[f / FN][f % FN][4 * g + 1], acc[f / FN][f % FN][4 * g + 2],
                            acc[f / FN][f % FN][4 * g + 3]};
    }
  __syncthreads();
  v16i sum[1][ON];
  if (owner) {
#pragma unroll
    for (int f = 0; f < FM * FN; ++f)                  // (registers have no index: the owner's fragments picked out)
      if (f / ON == wave) sum[0][f % ON] = acc[f / FN][f % FN];
#pragma unroll
    for (int o = 0; o < ON; ++o) {
      const int f = wave * ON + o;
#pragma unroll
      for (int w = 0; w < NW - 1; ++w) {
        const v4i* src = reinterpret_cast<const v4i*>(smem_all) + (f * (NW - 1) + w) * 256 + lane;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const v4i v = src[g * 64];
#pragma unroll
          for (int q = 0; q < 4; ++q) sum[0][o][4 * g + q] += v[q];
        }
      }
    }
    if (!CONV && __builtin_expect(p.corr_n != nullptr || p.corr_m != nullptr, 0)) {
      // zero points: sum (a - zx)(w - zw) = sum a w + corr_n[n] + corr_m[m] (as in qgemm_pipelined.h)
      const int m = m0 + wave * ON / FN * 32 + (lane & 31);
      const int cm = p.corr_m ? p.corr_m[m < p.M ? m : p.M - 1] : 0;
#pragma unroll
      for (int o = 0; o < ON; ++o)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int n = n0 + (wave * ON + o) % FN * 32 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4;
          sum[0][o][v] += cm + (p.corr_n ? p.corr_n[n < p.N ? n : p.N - 1] : 0);
        }
    }
  }
  constexpr bool kBlockStage = OWNERS == NW && (EPI == DQ8_EPI_REQUANT_CPU || EPI == DQ8_EPI_REQUANT_GPU);
  mfma_epilogue<EPI, 1, ON, NT, BN, NoHook, kBlockStage>(sum, p.epi, smem_all, m0 + wave * ON / FN * 32,
                                                         n0 + wave * ON % FN * 32, n0, col, wave, owner);
#else
  (void)p;
#endif
}

}  // namespace dq8

#endif  // DQ8_QGEMM_WAVE_H_
