// What kernels share whose blocks stay on the chip and hand results on in memory: room
// is filled with NONE first, results are written once, past the L2, and are never NONE.
#pragma once
#include "fei_common.h"

constexpr u32 NONE = 0xffffffffu;         // not there yet: two bfloat16 or a float32, NaN
constexpr int LIMIT = 1 << 20;            // looks

template <typename T> __device__ __forceinline__ T ld_sc(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A NaN of NONE's pattern becomes another.
__device__ __forceinline__ void st_sc(u32* p, u32 v) {
  __hip_atomic_store(p, v == NONE ? NONE - 1 : v, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u32 count(u32* p) {
  return __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Weights stay in flight, unlike at __syncthreads.
__device__ __forceinline__ void sync_lds() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ u32 raised(u32* flag) {
  return __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void raise(u32* flag) {
  __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Two results as a dword, by the hardware's conversion, round to nearest even.
__device__ __forceinline__ u32 pack(float x, float y) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  return __builtin_bit_cast(u32, __builtin_convertvector(f32x2{x, y}, bf16x2));
}
__device__ __forceinline__ float lo(u32 v) { return bf2f((u16)v); }
__device__ __forceinline__ float hi(u32 v) { return bf2f((u16)(v >> 16)); }

// A launch's state, in dwords, 0 at first. Blocks count themselves at the start. If all
// are there within 100 looks of any of them, each is bound to its items (FIXED), else
// items are taken by ticket, in order.
constexpr int ARRIVED = 0, HOW = 32, TICKET = 64, STATE = 96;
enum { FIXED = 1, TICKETS = 2 };
// A thread's: the block's number among ``blocks``, or NONE for tickets.
__device__ __forceinline__ u32 arrive(u32* state, int blocks) {
  const u32 r = count(state + ARRIVED);
  u32 how = 0;
  auto decide = [&](u32 to) {            // the first one does
    u32 none = 0;
    __hip_atomic_compare_exchange_strong(state + HOW, &none, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  };
  if (r == (u32)blocks - 1) decide(FIXED);
  for (int i = 0; (how = ld_sc(state + HOW)) == 0; ++i)
    if (i >= 100) decide(TICKETS);
  return how == FIXED ? r : NONE;
}
