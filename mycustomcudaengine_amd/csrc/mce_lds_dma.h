// Direct-to-LDS staging and the 32 x 32 matrix instruction, shared by the
// kernels that stream tiles through LDS.
#pragma once

#include "mce_common.h"

namespace mce {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Buffer descriptor word 3 for raw (stride 0) dword loads on gfx9-family
// parts: data format 32, no swizzle, range-checked against num_records.
constexpr int BUF_RSRC_WORD3 = 0x00020000;

// v_mfma_f32_32x32x16 on raw 16-bit operands of the element type.
template <class T>
__device__ __forceinline__ floatx16 mfma32(u32x4 a, u32x4 b, floatx16 c) {
  if constexpr (T::code == MCE_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a),
                                                  __builtin_bit_cast(half8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Buffer load of 16 bytes per lane straight into LDS: lane l's bytes land at
// LDS address m0 + 16 l (m0 wave-uniform).  Written as inline asm rather than
// the builtin: the compiler orders the builtin's LDS write before every later
// read of the same LDS array with a vmcnt wait, which would stall the step's
// fragment reads (of the other buffer) until the load landed.  The waits the
// kernel needs are explicit (s_waitcnt vmcnt before the publishing barrier);
// loads the compiler does not see only make its own vmcnt waits stricter.
// The asm also carries the wait state that gfx9-family parts need between a
// scalar write of M0 (which the constraint produces just before it) and an
// LDS-DMA load: the compiler inserts it before the builtin but cannot insert
// it into inline asm.  (The scalar offset must come from scalar code or a
// constant: a v_readfirstlane result would need five more wait states.)
// NT: with the non-temporal policy (bytes that are used once).
template <bool NT = false>
__device__ __forceinline__ void buffer_load_lds16(i32x4 rsrc, int voff, int soff, unsigned m0) {
  if constexpr (NT)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds" : : "v"(voff), "s"(rsrc),
                 "s"(soff), "{m0}"(m0));
  else
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(voff), "s"(rsrc),
                 "s"(soff), "{m0}"(m0));
}

// Raw buffer descriptor (stride 0, range-checked against `bytes`).
__device__ inline i32x4 buffer_rsrc(const void *base, int bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  return i32x4{(int)(uint32_t)p, (int)(uint32_t)(p >> 32) & 0xffff, bytes, BUF_RSRC_WORD3};
}

// s_waitcnt vmcnt(N): all but the wave's N youngest loads have landed (loads
// complete in issue order).
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

}  // namespace mce
