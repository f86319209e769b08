// What the GEMMs with operands straight into LDS share (rows_gemm.hip,
// wide_gemm.hip).
#pragma once

#include "lm_common.h"

using rsrc_t = __amdgpu_buffer_rsrc_t;
typedef __attribute__((address_space(3))) void lds_void_t;

// of the products as they are stored, or of their sums
enum { ACT_NONE = 0, ACT_SILU = 1, ACT_GELU = 2, ACT_SILU_SUM = 3 };

__device__ __forceinline__ float as_bf16(float v) {
  return bf16_to_f32(cvt_bf16(v));
}

// all of a wave's LDS reads are in, and at most N of its loads under way
template <int N> __device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "the counter's range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | 7 << 4);
}

// A barrier that neither waits for loads nor lets memory accesses pass: what
// the waves have read and received is settled by wait_loads before it.
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}
