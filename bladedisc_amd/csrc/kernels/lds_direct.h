// Loads that go from memory straight into LDS (gfx950), and the waits for them: shared by the
// int8 GEMM and convolution kernels and the weight-only GEMM.
#ifndef DQ8_LDS_DIRECT_H_
#define DQ8_LDS_DIRECT_H_

#include <hip/hip_runtime.h>

#include <cstdint>

namespace dq8 {

typedef int v4i __attribute__((ext_vector_type(4)));

// gfx9 raw buffer descriptor word 3: 32-bit data format, no swizzle
constexpr int kBufferRsrcWord3 = 0x00020000;

typedef __attribute__((address_space(3))) void lds_void_t;

// 128-bit raw buffer descriptor (stride 0): base address, byte count, format word.  The
// descriptor is a scalar operand of the load: base and size are the same in every lane, and
// the readfirstlane says so where the compiler cannot see it (it folds away where it can).
__device__ __forceinline__ v4i make_rsrc(const void* base, int64_t num_records) {
  const uint64_t b = (uint64_t)base;
  v4i r = {__builtin_amdgcn_readfirstlane((int)(uint32_t)b),
           __builtin_amdgcn_readfirstlane((int)(uint32_t)((b >> 32) & 0xffff)),
           __builtin_amdgcn_readfirstlane((int)num_records), kBufferRsrcWord3};
  return r;
}

// One 16-byte-per-lane buffer load whose result goes straight to LDS: lane i's
// data lands at lds_addr + 16*i (lds_addr is wave-uniform and goes through M0).
// Issued as inline assembly so that the wave decides itself, with an explicit
// s_waitcnt vmcnt, when it needs the data; through the compiler builtin every LDS
// read would first wait for all loads in flight.
__device__ __forceinline__ void buffer_load_lds_b128(v4i rsrc, unsigned lds_addr, int voffset) {
  // (wave-uniform by construction; said explicitly for where the compiler cannot prove it)
  lds_addr = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
#pragma unroll
  for (int c = 0; c < 4; ++c) rsrc[c] = __builtin_amdgcn_readfirstlane(rsrc[c]);
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, 0 offen lds"
      :
      : "s"(lds_addr), "v"(voffset), "s"(rsrc)
      : "memory", "m0");
}

// The same with 4 bytes per lane, lane i's at lds_addr + 4 i.
__device__ __forceinline__ void buffer_load_lds_b32(v4i rsrc, unsigned lds_addr, int voffset) {
  lds_addr = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
#pragma unroll
  for (int c = 0; c < 4; ++c) rsrc[c] = __builtin_amdgcn_readfirstlane(rsrc[c]);
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dword %1, %2, 0 offen lds"
      :
      : "s"(lds_addr), "v"(voffset), "s"(rsrc)
      : "memory", "m0");
}

// The last chunk of rows of K bytes (K % 4 == 0, not a multiple of 16), loaded as the last 16 bytes of the row:
// the words that belong to the chunk before it set to zero.  A fragment of 32 bytes of k has the chunk in the lanes of half
// (K / 16) % 2 of the wave.
__device__ __forceinline__ void clear_row_end(v4i& fragment, int K, int lane) {
  const int drop = (lane >> 5) == ((K >> 4) & 1) ? 4 - ((K >> 2) & 3) : 0;
#pragma unroll
  for (int c = 0; c < 3; ++c) fragment[c] = c < drop ? 0 : fragment[c];
}

// s_waitcnt immediate for gfx9: vmcnt = n (6 bits, split), lgkmcnt = 0, expcnt = any
constexpr int waitcnt_vm_lgkm0(int n) { return (n & 0xf) | ((n >> 4) << 14) | (0x7 << 4); }

}  // namespace dq8

#endif  // DQ8_LDS_DIRECT_H_
