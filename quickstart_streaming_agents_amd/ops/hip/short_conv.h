// Device code of the short convolutions (short_conv.hip) that other kernels of a
// decoding step share.
#pragma once

#include <type_traits>

#include "lm_common.h"
#include "step_args.h"

#define CONV_ROWS 16  // tokens per thread; taps - 1 must not exceed it

struct ConvSpan { int r0, t0, t1, n, p0, slot; };

// The rows of chunk c, or of one of the `parts` that share them: as short as a filter is
// long, so that still only the first of a portion looks at the tail.
#define CONV_PARTS 4
__device__ __forceinline__ ConvSpan conv_span(const ConvStep& st, int c,
                                              int part = 0, int parts = 1) {
  ConvSpan s;
  if (st.item) {
    const int it = st.item[c], rows = CONV_ROWS / parts;
    s.r0 = st.off[it];
    s.t0 = st.t0[c] + part * rows;
    s.n = st.len[it];
    s.p0 = st.start[it];
    s.slot = st.slots[it];
    s.t1 = min(s.t0 + rows, s.n);
  } else {
    s.r0 = c;
    s.t0 = 0;
    s.n = s.t1 = 1;
    s.p0 = st.start[c] - 1;
    s.slot = st.slots[c];
  }
  return s;
}

// NP (1 or 2) groups of VEC channels, c0.. and c1..; TAPS 0: `taps` of them,
// through memory.  pre(t) loads what emit(t, values, .) wants besides.
// SINGLE: tokens one by one, which takes fewer registers (conv_single, short_conv.hip).
template <typename T, int TAPS, int VEC, int NP, bool SINGLE, typename Pre,
          typename Emit>
__device__ __forceinline__ void conv_rows(
    const T* x, long long xstride, T* tail, int C, int c0, int c1,
    const float* w, const float* bias, int taps, const ConvSpan& s, Pre pre,
    Emit emit) {
  const int NT = (TAPS ? TAPS : taps) - 1;
  auto ch = [&](int p) { return p == 0 ? c0 : c1; };
  // few blocks: chosen by address, as a branch for each would wait for each
  auto load = [&](int t, int p, float* v) {
    if constexpr (SINGLE) {
      if (t >= 0) {
        ldv<T, VEC>(x + (long long)(s.r0 + t) * xstride + ch(p), v);
      } else if (s.p0 + t >= 0) {
        ldv<T, VEC>((const T*)tail + (long long)(NT + t) * C + ch(p), v);
      } else {
#pragma unroll
        for (int i = 0; i < VEC; ++i) v[i] = 0.f;
      }
      return;
    }
    const T* at = t >= 0 ? x + (long long)(s.r0 + t) * xstride
                         : (const T*)tail + (long long)(NT + t) * C;
    ldv<T, VEC>(at + ch(p), v);
    const bool none = s.p0 + t < 0;
#pragma unroll
    for (int i = 0; i < VEC; ++i) v[i] = none ? 0.f : v[i];
  };
  float b[NP][VEC];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    if (bias) {
      ldv<float, VEC>(bias + ch(p), b[p]);
    } else {
#pragma unroll
      for (int i = 0; i < VEC; ++i) b[p][i] = 0.f;
    }
  }
  if constexpr (TAPS > 0) {
    constexpr int K = TAPS > 1 ? TAPS - 1 : 1;
    float wt[NP][TAPS][VEC], win[NP][K][VEC];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int j = 0; j < TAPS; ++j)
        ldv<float, VEC>(w + (long long)j * C + ch(p), wt[p][j]);
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j)
        load(s.t0 - (TAPS - 1) + j, p, win[p][j]);
    }
    auto step = [&](int t, const float (&u)[NP][VEC], const auto& aux) {
      float a[NP][VEC];
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
          a[p][i] = b[p][i];
#pragma unroll
          for (int k = 0; k < TAPS - 1; ++k)
            a[p][i] = fmaf(wt[p][k][i], win[p][k][i], a[p][i]);
          a[p][i] = fmaf(wt[p][TAPS - 1][i], u[p][i], a[p][i]);
#pragma unroll
          for (int k = 0; k + 2 < TAPS; ++k) win[p][k][i] = win[p][k + 1][i];
          win[p][K - 1][i] = u[p][i];
        }
      emit(t, a, aux);
    };
    // All loads of AHEAD tokens go out before the first of them is used: a store may
    // write what a later load reads, as far as the compiler knows, so in one loop each
    // token waited for memory by itself.  4096 channels with four taps, to pages / with
    // silu, us: 60 tokens 15.2 / 10.8 -> 9.9 / 7.7 (to pages two and four tokens ahead
    // were 13.2 and 10.6), 7500 with silu 40.2 -> 33.8.
    auto walk = [&](auto ahead) {
      constexpr int AHEAD = ahead.value;
      for (int t0 = s.t0; t0 < s.t1; t0 += AHEAD) {
        float u[AHEAD][NP][VEC];
        decltype(pre(0)) aux[AHEAD];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
          const int t = min(t0 + j, s.t1 - 1);
#pragma unroll
          for (int p = 0; p < NP; ++p)
            ldv<T, VEC>(x + (long long)(s.r0 + t) * xstride + ch(p), u[j][p]);
          aux[j] = pre(t);
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
          if (t0 + j >= s.t1) break;              // uniform over the block
          step(t0 + j, u[j], aux[j]);
        }
      }
    };
    if constexpr (SINGLE) {
#pragma unroll 4
      for (int t = s.t0; t < s.t1; ++t) {
        const auto aux = pre(t);
        float u[NP][VEC];
#pragma unroll
        for (int p = 0; p < NP; ++p)
          ldv<T, VEC>(x + (long long)(s.r0 + t) * xstride + ch(p), u[p]);
        step(t, u, aux);
      }
    } else if (s.t1 - s.t0 == 1) walk(std::integral_constant<int, 1>{});
    else if (s.t1 - s.t0 <= CONV_ROWS / CONV_PARTS)
      walk(std::integral_constant<int, CONV_ROWS / CONV_PARTS>{});
    else walk(std::integral_constant<int, NP == 1 && sizeof(T) == 2 ? 16 : 8>{});
    if (s.t0 == 0) {
      // The new tail: of a whole portion, as of a single token, the window, else the
      // portion's last rows, all of them read before one is written (moving entries
      // in memory takes a round trip each: 64 single tokens, four taps, 4096 channels
      // to pages 8.7 us, 7.5 so, dense 5.8, 5.1).
      if (s.t1 != s.n)
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j)
#pragma unroll
          for (int p = 0; p < NP; ++p) load(s.n - NT + j, p, win[p][j]);
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j)
#pragma unroll
        for (int p = 0; p < NP; ++p)
          stv<T, VEC>(tail + (long long)j * C + ch(p), win[p][j]);
    }
    return;
  } else {
    for (int t = s.t0; t < s.t1; ++t) {
      const auto aux = pre(t);
      float a[NP][VEC];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) a[p][i] = b[p][i];
        for (int j = 0; j <= NT; ++j) {
          float u[VEC], wj[VEC];
          load(t - NT + j, p, u);
          ldv<float, VEC>(w + (long long)j * C + ch(p), wj);
#pragma unroll
          for (int i = 0; i < VEC; ++i) a[p][i] = fmaf(wj[i], u[i], a[p][i]);
        }
      }
      emit(t, a, aux);
    }
  }
  if (s.t0 == 0) {
    // entry j moves from n + j, never from a place already overwritten
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        float v[VEC];
        load(s.n - NT + j, p, v);
        stv<T, VEC>(tail + (long long)j * C + ch(p), v);
      }
  }
}

#define CONV_CASE(T, TAPS, VEC, NP)                                          \
  conv_rows<T, TAPS, VEC, NP, SINGLE>(x, xstride, tail, C, c0, c1, w, bias,  \
                                      taps, s, pre, emit)
#define CONV_DISPATCH(T, VEC, NP)              \
  switch (taps) {                              \
    case 1: CONV_CASE(T, 1, VEC, NP); break;   \
    case 2: CONV_CASE(T, 2, VEC, NP); break;   \
    case 3: CONV_CASE(T, 3, VEC, NP); break;   \
    case 4: CONV_CASE(T, 4, VEC, NP); break;   \
    default: CONV_CASE(T, 0, VEC, NP);         \
  }

template <int VEC>
struct Turn {
  int slot;                    // where k or v goes
  float c[VEC], s[VEC];
};

// A thread owns a pair of channel groups: of q and k a rotated pair (i,
// i + rot/2) or two groups behind the rotated ones, of v two groups.
// Pages: k [pages, G, 64, D], v [pages, G, 64, E].
// units of a row
__host__ __device__ inline int conv_qkv_units(const ConvQkv& p, int vec) {
  return (p.H + p.G) * (p.rot / 2 / vec +
                        (p.D - p.rot + 2 * vec - 1) / (2 * vec)) +
         p.G * ((p.E + 2 * vec - 1) / (2 * vec));
}

// ONE: the step has one token per row and filters of up to CONV_ONE_TAPS taps
#define CONV_ONE_TAPS 4
template <typename T, int VEC, bool ONE = false, bool SINGLE = false>
__device__ __forceinline__ void conv_qkv_unit(const ConvQkv& p, int chunk,
                                              int u, int part = 0,
                                              int parts = 1) {
  const T* x = (const T*)p.x;
  const long long xstride = p.xstride;
  const float* __restrict__ w = p.w;
  const int taps = p.taps, rot = p.rot, H = p.H, G = p.G, D = p.D, E = p.E;
  const float* __restrict__ cos_t = p.cos_t;
  const float* __restrict__ sin_t = p.sin_t;
  const int table_len = p.table_len;
  T *q = (T*)p.q, *kc = (T*)p.kc, *vc = (T*)p.vc;
  const int half = rot >> 1;
  const int ur = half / VEC, up = (D - rot + 2 * VEC - 1) / (2 * VEC);
  const int ud = ur + up, ue = (E + 2 * VEC - 1) / (2 * VEC);
  if (u >= (H + G) * ud + G * ue) return;
  ConvSpan s;
  if constexpr (ONE)
    s = {chunk, 0, 1, 1, p.step.start[chunk] - 1, p.step.slots[chunk]};
  else
    s = conv_span(p.step, chunk, part, parts);
  if (s.slot < 0 || s.p0 < 0 || s.t0 >= s.n) return;
  const int C = (H + G) * D + G * E;
  T* tail = (T*)p.tails + (long long)s.slot * (taps - 1) * C;
  const float* bias = nullptr;
  const bool val = u >= (H + G) * ud;
  const int un = val ? ue : ud;
  const int r = (val ? u - (H + G) * ud : u) % un;
  const int head = (val ? u - (H + G) * ud : u) / un;
  const bool turn = !val && r < ur;
  const int d0 = val || turn ? r * VEC : rot + (r - ur) * VEC;
  const int far = d0 + (val ? ue * VEC : turn ? half : up * VEC);
  const bool two = far < (val ? E : D);
  const int d1 = two ? far : d0;
  const int base = val ? (H + G) * D + head * E : head * D;
  const int c0 = base + d0, c1 = base + d1;
  const bool query = !val && head < H;
  // chosen here: in the closures below they would be chosen by address, in memory
  T* const to = query ? q : val ? vc : kc;
  const int page_head = val ? head : head - H, width = val ? E : D;
  // a block's tokens are the same for all its threads: scalar loads
  const auto page_slots =
      (const __attribute__((address_space(4))) int*)p.cache_slots;
  auto pre = [=](int t) {
    Turn<VEC> r;
    r.slot = page_slots[s.r0 + t];
    if (turn) {
      const long long at =
          (long long)min(s.p0 + t, table_len - 1) * half + d0;
      ldv<float, VEC>(cos_t + at, r.c);
      ldv<float, VEC>(sin_t + at, r.s);
    }
    return r;
  };
  auto emit = [=](int t, float (&a)[2][VEC], const Turn<VEC>& r) {
    if (turn) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        // fused here, not as the compiler likes, so that every form of a step
        // leaves the same bits
        const float u0 = a[0][i], v0 = a[1][i];
        a[0][i] = fmaf(u0, r.c[i], -(v0 * r.s[i]));
        a[1][i] = fmaf(u0, r.s[i], v0 * r.c[i]);
      }
    }
    if (!query && r.slot < 0) return;
    const long long in_pages =
        ((long long)(r.slot >> 6) * G + page_head) * 64 + (r.slot & 63);
    const long long in_rows = (long long)(s.r0 + t) * H + head;
    T* const dst = to + (query ? in_rows : in_pages) * width;
    stv<T, VEC>(dst + d0, a[0]);
    if (two) stv<T, VEC>(dst + d1, a[1]);
  };
  if constexpr (ONE) {
    switch (taps) {
      case 1: CONV_CASE(T, 1, VEC, 2); break;
      case 2: CONV_CASE(T, 2, VEC, 2); break;
      case 3: CONV_CASE(T, 3, VEC, 2); break;
      case 4: CONV_CASE(T, 4, VEC, 2); break;
    }
  } else {
    CONV_DISPATCH(T, VEC, 2)
  }
}
