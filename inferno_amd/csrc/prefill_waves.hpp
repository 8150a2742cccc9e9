// Pieces of the kernels whose waves share rows or stage by hand
// (prefill_narrow.hip, prefill_pair.hip, sparse.hip): lane-pair exchanges, loads into LDS
// with written-out waits, and the barrier that leaves loads in flight.
#pragma once

#include "prefill_common.hpp"

namespace ifr {
namespace prefill {

// Members of the (lane, lane ^ 16) and (lane, lane ^ 32) pairs, lower lane
// first, the same in both lanes.
__device__ __forceinline__ void pair16(float x, float& lo, float& hi) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}
__device__ __forceinline__ void pair32(float x, float& lo, float& hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}
__device__ __forceinline__ float raw_max(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// Over the four 16-lane groups.
__device__ __forceinline__ float groups_max(float x) {
  float a, b;
  pair16(x, a, b);
  x = raw_max(a, b);
  pair32(x, a, b);
  return raw_max(a, b);
}
__device__ __forceinline__ float groups_mul(float x) {
  float a, b;
  pair16(x, a, b);
  x = a * b;
  pair32(x, a, b);
  return a * b;
}
__device__ __forceinline__ float groups_add(float x) {
  float a, b;
  pair16(x, a, b);
  x = a + b;
  pair32(x, a, b);
  return a + b;
}

// 1 KiB loads into LDS: load i goes to lds (wave-uniform) + 1024 i + 16 * lane,
// from base (wave-uniform) + off_i + 1024 i (the instruction's offset counts on
// both sides; off_i is unsigned, so callers keep base low enough).  As
// instructions the compiler does not track: its tracking of such loads stops at
// the transposing LDS reads, which carry no alias information, and would wait
// there for every load in flight.  The waits are written out below (loads return
// in order, so the ones the compiler adds for its own loads can only wait for
// more).  m0 is put back, as the compiler does not know of the change; a write of m0
// needs one wait state before a load that reads it.
__device__ __forceinline__ uint32_t lds_addr(const uint8_t* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_t*)p));
}
__device__ __forceinline__ void load_lds4(const char* base, uint32_t o0, uint32_t o1, uint32_t o2,
                                          uint32_t o3, const uint8_t* lds) {
  uint32_t m0;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t"
      "global_load_lds_dwordx4 %2, %6\n\t"
      "global_load_lds_dwordx4 %3, %6 offset:1024\n\t"
      "global_load_lds_dwordx4 %4, %6 offset:2048\n\t"
      "global_load_lds_dwordx4 %5, %6 offset:3072\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(m0)
      : "s"(lds_addr(lds)), "v"(o0), "v"(o1), "v"(o2), "v"(o3), "s"(base)
      : "memory");
}
__device__ __forceinline__ void load_lds2(const char* base, uint32_t o0, uint32_t o1,
                                          const uint8_t* lds) {
  uint32_t m0;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t"
      "global_load_lds_dwordx4 %2, %4\n\t"
      "global_load_lds_dwordx4 %3, %4 offset:1024\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(m0)
      : "s"(lds_addr(lds)), "v"(o0), "v"(o1), "s"(base)
      : "memory");
}

// Waits until at most n loads are outstanding.  The memory clobber keeps the LDS
// reads of what they bring behind it.
template <int n>
__device__ __forceinline__ void wait_loads() {
  if constexpr (n == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else if constexpr (n == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else if constexpr (n == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  else if constexpr (n == 16) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  else static_assert(n == 0, "a count with an instruction");
}

// LDS written so far is visible to the block; the loads in flight stay in
// flight (a __syncthreads would wait for them).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace prefill
}  // namespace ifr
