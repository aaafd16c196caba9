// What products of a few rows with a weight matrix share (rows_gemm.hip for
// bf16 weights, rows_quant.hip for GGUF blocks).
#pragma once

#include "common.h"

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((ext_vector_type(4))) float float4v;

#define LDS_LOAD_ARGS(g, lds)                                        \
  (const __attribute__((address_space(1))) unsigned int*)(g),        \
      (__attribute__((address_space(3))) unsigned int*)(lds)

// SZ bytes of every lane go from its address to lds + lane * SZ.
template <int SZ>
DEV_INLINE void load_to_lds(const void* g, void* lds) {
  static_assert(SZ == 16 || SZ == 4);
  if constexpr (SZ == 16)
    __builtin_amdgcn_global_load_lds(LDS_LOAD_ARGS(g, lds), 16, 0, 0);
  else
    __builtin_amdgcn_global_load_lds(LDS_LOAD_ARGS(g, lds), 4, 0, 0);
}

// Until no more than the N loads issued last are in flight.
template <int N>
DEV_INLINE void wait_loads() {
  static_assert(N < 64);
  asm volatile("s_waitcnt vmcnt(%0)" :: "i"(N) : "memory");
}

// What was read from LDS is in registers: its place may be loaded over.
DEV_INLINE void wait_lds_reads() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// The weight row behind row r of the 16 that a workgroup from column n0 on
// multiplies. Gated: eight of the gates, then the same eight of what they
// gate, whose rows begin halfway.
template <bool GATED>
DEV_INLINE int weight_row(int n0, int r, int n) {
  if constexpr (GATED) return n0 + (r & 7) + (r >> 3) * (n / 2);
  return min(n0 + r, n - 1);
}

DEV_INLINE float silu_times(float g, float u) {
  return g / (1.f + __expf(-g)) * u;
}
