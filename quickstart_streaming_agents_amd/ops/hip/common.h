// Shared device helpers for the qsa MI355X (gfx950) kernels.
// Wave width is 64 on CDNA4 — hard-coded per the platform guide.
#pragma once

#include <hip/hip_runtime.h>

#define QSA_WAVE 64

// The last-level cache, and the cache policy of loads through buffers or to LDS that
// leave no trace in it (__builtin_nontemporal_load otherwise).  What is read once
// in a step whose reads do not fit there together only drives out the rest.
#define QSA_LLC (256ll << 20)
#define QSA_NT 2
// keys and values of one layer, in bytes, beyond which a step reads them so
#define QSA_FAR_PAGES (32ll << 20)

// ---- bf16 <-> f32 ----------------------------------------------------------
__device__ __forceinline__ float bf16_to_f32(unsigned short h) {
  union { unsigned int u; float f; } v;
  v.u = ((unsigned int)h) << 16;
  return v.f;
}

// Round to nearest even, NaN stays NaN, with the hardware's packed conversion.  In
// integer operations it was two branches a value: the rotation of a decoding
// step's query and key alone 1400 instructions of a wave, now 190.
__device__ __forceinline__ unsigned int f32x2_to_bf16x2(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) float f2;
  typedef __attribute__((ext_vector_type(2))) __bf16 b2;
  return __builtin_bit_cast(unsigned int,
                            __builtin_convertvector((f2){a, b}, b2));
}

__device__ __forceinline__ unsigned short f32_to_bf16(float f) {
  return __builtin_bit_cast(unsigned short, (__bf16)f);
}

// unpack 2 bf16 held in one uint (lo, hi)
__device__ __forceinline__ float2 bf16x2_to_f32x2(unsigned int p) {
  union { unsigned int u; float f; } lo, hi;
  lo.u = p << 16;
  hi.u = p & 0xffff0000u;
  return make_float2(lo.f, hi.f);
}

// ---- wave reductions (64-lane) --------------------------------------------
// Reductions over lanes by exchanges between registers: __shfl_xor goes through
// LDS, some 100 cycles a step that a chain of six waits for.  Every lane ends up
// with the value, in the order of a butterfly of steps 32, 16, 8, 4, 2, 1: behind
// a step the lanes that the later ones tell apart are all that differ, so turning
// a row of 16 is as good as crossing lanes (sums of two do not mind their order).
template <int CTRL>
__device__ __forceinline__ float qsa_dpp(float v) {
  const int x = __float_as_int(v);
  return __int_as_float(
      __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false));
}
#define QSA_ROW_TURN 0x120             // + lanes
#define QSA_ROW_MIRROR 0x140           // lane i of a row from 15 - i
#define QSA_HALF_MIRROR 0x141          // ... of half a row from 7 - i
#define QSA_QUAD_1 0xb1                // lane i from i ^ 1
#define QSA_QUAD_2 0x4e                // ... i ^ 2

// f(v of lane i, v of lane i ^ 16), and 32
template <class F>
__device__ __forceinline__ float qsa_cross16(float v, F f) {
  const auto r = __builtin_amdgcn_permlane16_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <class F>
__device__ __forceinline__ float qsa_cross32(float v, F f) {
  const auto r = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

struct QsaAdd {
  __device__ float operator()(float a, float b) const { return a + b; }
};
struct QsaMax {
  __device__ float operator()(float a, float b) const { return fmaxf(a, b); }
};

// over the four lanes that share a lane's place in its row of 16
template <class F>
__device__ __forceinline__ float qsa_over_rows(float v, F f) {
  return qsa_cross32(qsa_cross16(v, f), f);
}
__device__ __forceinline__ float rows_sum(float v) {
  return qsa_over_rows(v, QsaAdd());
}
__device__ __forceinline__ float rows_max(float v) {
  return qsa_over_rows(v, QsaMax());
}

// over a row of 16, in steps 1, 2, 4, 8
__device__ __forceinline__ float row16_sum(float v) {
  v += qsa_dpp<QSA_QUAD_1>(v);
  v += qsa_dpp<QSA_QUAD_2>(v);
  v += qsa_dpp<QSA_HALF_MIRROR>(v);
  return v + qsa_dpp<QSA_ROW_MIRROR>(v);
}

template <class F>
__device__ __forceinline__ float qsa_over_wave(float v, F f) {
  v = qsa_cross16(qsa_cross32(v, f), f);
  v = f(v, qsa_dpp<QSA_ROW_TURN + 8>(v));
  v = f(v, qsa_dpp<QSA_ROW_TURN + 4>(v));
  v = f(v, qsa_dpp<QSA_ROW_TURN + 2>(v));
  return f(v, qsa_dpp<QSA_ROW_TURN + 1>(v));
}
__device__ __forceinline__ float wave_reduce_sum(float v) {
  return qsa_over_wave(v, QsaAdd());
}
__device__ __forceinline__ float wave_reduce_max(float v) {
  return qsa_over_wave(v, QsaMax());
}

// Sum over n numbers of what `of` makes of them, in every lane (all lanes on): what a
// launch has before it, where only the device knows.  Up to 256 numbers are loads
// side by side, beside those that a kernel begins with.
template <class F>
__device__ __forceinline__ float wave_total(const int* at, int n, F of) {
  constexpr int U = 4;
  float v = 0.f;
  for (int i = threadIdx.x & 63; i < n; i += U * QSA_WAVE) {
    int x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = at[min(i + u * QSA_WAVE, n - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u * QSA_WAVE < n) v += of(x[u]);
  }
  return __int_as_float(
      __builtin_amdgcn_readfirstlane(__float_as_int(wave_reduce_sum(v))));
}

// Exchanges of two words at once, for the better of two (value, place) pairs:
// better(other value, other place, value, place).
template <int CTRL, class B>
__device__ __forceinline__ void qsa_dpp_best(float& v, int& i, B better) {
  const float ov = qsa_dpp<CTRL>(v);
  const int oi = __builtin_amdgcn_update_dpp(i, i, CTRL, 0xf, 0xf, false);
  if (better(ov, oi, v, i)) {
    v = ov;
    i = oi;
  }
}
// the best of a row of 16, in all its lanes
template <class B>
__device__ __forceinline__ void row16_best(float& v, int& i, B better) {
  qsa_dpp_best<QSA_QUAD_1>(v, i, better);
  qsa_dpp_best<QSA_QUAD_2>(v, i, better);
  qsa_dpp_best<QSA_HALF_MIRROR>(v, i, better);
  qsa_dpp_best<QSA_ROW_MIRROR>(v, i, better);
}
template <class B>
__device__ __forceinline__ void wave_best(float& v, int& i, B better) {
  row16_best(v, i, better);
  auto pick = [&](auto a, auto b) {
    const float x = __uint_as_float(a[0]), y = __uint_as_float(a[1]);
    const int p = (int)b[0], q = (int)b[1];
    const bool second = better(y, q, x, p);
    v = second ? y : x;
    i = second ? q : p;
  };
  pick(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v),
                                        false, false),
       __builtin_amdgcn_permlane16_swap((unsigned)i, (unsigned)i, false,
                                        false));
  pick(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v),
                                        false, false),
       __builtin_amdgcn_permlane32_swap((unsigned)i, (unsigned)i, false,
                                        false));
}

// Block reduction via LDS (callers pass scratch of >= nwaves floats).
// All threads receive the result.
__device__ __forceinline__ float block_reduce_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (QSA_WAVE - 1);
  const int wave = threadIdx.x / QSA_WAVE;
  const int nwaves = blockDim.x / QSA_WAVE;
  v = wave_reduce_sum(v);
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll 4
  for (int i = 0; i < nwaves; ++i) total += scratch[i];
  __syncthreads();
  return total;
}

#define QSA_CHECK(cond, msg)                                            \
  TORCH_CHECK(cond, "qsa_hip: ", msg)

typedef __attribute__((ext_vector_type(2))) __bf16 qsa_bf16x2_t;
__device__ __forceinline__ qsa_bf16x2_t as_bf16x2(unsigned int u) {
  union { unsigned int u; qsa_bf16x2_t v; } c;
  c.u = u;
  return c.v;
}
