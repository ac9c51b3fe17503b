// Shared helpers for the gfx950 kernels of the paged-attention path.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "auto_infer_amd.h"

namespace aia {

// Records a message for aia_last_error() (thread local) and returns `code`.
int fail(int code, const char* fmt, ...);
// Maps a HIP status to AIA_ERR_HIP with the runtime's message.
int check_hip(hipError_t err, const char* what);

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// bf16 <- f32, round to nearest even (inputs here are finite).
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// Two floats -> packed bf16 pair, round to nearest even (gfx950 converts a
// pair in one instruction, v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// Reductions over lanes l, l^16, l^32, l^48 (the 4 lane groups of an MFMA
// 16-row fragment) with gfx950's VALU lane swaps instead of ds_bpermute's
// LDS crossbar round trip.  Given the same value in both operands,
// v_permlane16_swap / v_permlane32_swap leave each lane holding x[l] and
// x[l ^ 16] (resp. x[l ^ 32]) in its two results, so max or sum of the pair
// equals the xor-shuffle step bit for bit (both operations commute).
__device__ __forceinline__ float group4_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// The same over lanes l and l ^ 32 (the 2 lane groups of a 32-row fragment).
__device__ __forceinline__ float group2_max(float x) {
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float group2_sum(float x) {
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ float group4_sum(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// One 16-byte direct load from global memory into LDS at byte lds + 16 lane
// (lds wave-uniform).  Issued as inline assembly on purpose: the compiler's
// counter-wait pass tracks the builtin form as an outstanding LDS access and
// then waits for the LDS counter to drain completely (lgkmcnt(0)) before
// every LDS read, which exposes each read's full latency (the GQA prefill
// units, us per call: 49.3 with the builtin against 48.2, and 47.6-47.9
// against 46.0 with V read from LDS ahead of its use).  Completion is explicit
// instead: a wave waits for its own loads (s_waitcnt vmcnt) before the barrier
// that publishes their bytes.  Loads the compiler does not see can only make
// its own vmcnt waits stricter, never too weak (the counter retires in order).
// m0 (the LDS address of the load) is named as clobbered, which clang warns
// about for a register it reserves: the warning is silenced here because the
// clobber is what tells the compiler that m0 changed, and the compiler keeps
// no value of its own in m0 in these kernels (their device assembly sets m0
// only in front of these loads).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_load16(const uint16_t* src, uint16_t* lds) {
  const uint32_t la = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(la), "v"(src) : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// s_waitcnt vmcnt(0) (expcnt / lgkmcnt left at their maxima), gfx9 encoding:
// what a lds_load16 needs before the barrier that publishes its bytes.
constexpr int kWaitVmcnt0 = 0x0F70;

}  // namespace aia
