// Attention of the retrieval encoder for CDNA4 (gfx950): every token of an
// item sees every other, q, k and v are the projection's rows.
//
// Items are short (some 100 tokens, 512 at most), so nothing is laid out between
// the projection and here: a block (64 query rows of an item, head) rotates its
// queries in registers and the keys on their way to LDS, 64 at a time, where the
// values keep their rows for the transposing read.  A wave has 16 rows; scores
// come out transposed (row = key, column = query), so softmax state and weights
// are lane-local.  Vector work and latencies bound it: hidden keys are looked
// for in the last tile only, the scale joins the exponent in one fma, and four
// blocks fit a CU (128 rows and keys a block rotate each key fewer times, but
// one block fits: 30 us).
// 64 items of 137 tokens, 8 heads of 64: rotation into pages and attention over
// them 13.4 + 17.6 us as two kernels, 19.2 us here (20.2 with the last tile's
// 16s of keys without a key computed as well).  A block per item that has all keys
// in LDS once, and heads of an item on one die, were no faster.
#include <type_traits>

#include "lm_common.h"

#define ENC_KEYS 64

// rotate dims d.. and d + D/2.. of a row, rounded to bf16
__device__ __forceinline__ void enc_rotate(u32x4_v& a, u32x4_v& b,
                                           const float* c, const float* s) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float2 x = bf16x2_to_f32x2(a[e]), y = bf16x2_to_f32x2(b[e]);
    const float* ce = c + 2 * e;
    const float* se = s + 2 * e;
    a[e] = cvt_bf16x2(x.x * ce[0] - y.x * se[0], x.y * ce[1] - y.y * se[1]);
    b[e] = cvt_bf16x2(x.x * se[0] + y.x * ce[0], x.y * se[1] + y.y * ce[1]);
  }
}

template <int D>
__global__ void __launch_bounds__(256, D == 64 ? 4 : 2)
qsa_encoder_attn(const bf16_t* __restrict__ qkv,      // [T, 3, H, D]
                 const float* __restrict__ cos_t,     // [positions, D/2]
                 const float* __restrict__ sin_t, int positions,
                 const int* __restrict__ qb_item,     // [blocks of 64 rows]
                 const int* __restrict__ qb_t0,
                 const int* __restrict__ off,         // [items] first row
                 const int* __restrict__ len,         // [items]
                 bf16_t* __restrict__ out,            // [T, H, D]
                 int H, float scale2) {
  constexpr int KS = D / 32, ET = D / 16;
  constexpr int KP = D + 8, VP = D + 16;              // LDS pitches
  constexpr int LT = D / 16, TB = 256 / LT, NP = ENC_KEYS / TB;
  __shared__ __attribute__((aligned(16))) bf16_t kt[ENC_KEYS * KP];
  __shared__ __attribute__((aligned(16))) bf16_t vt[ENC_KEYS * VP];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  const int h = blockIdx.x % H, qb = blockIdx.x / H;
  const int item = qb_item[qb], t0 = qb_t0[qb];
  const int n = len[item];
  if (n <= 0 || t0 >= n) return;       // uniform over the block
  const long long A = (long long)H * D, r0 = off[item];
  const bf16_t* base = qkv + r0 * 3 * A + (long long)h * D;
  const int w0 = t0 + wave * 16;       // first row of this wave

  // a lane takes 8 dims and their partners of a key
  const int d = (tid % LT) * 8;
  u32x4_v kx[NP], ky[NP], vx[NP], vy[NP];
  float c[NP][8], s[NP][8];
  auto fetch = [&](int tile) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int key = min(tile * ENC_KEYS + p * TB + tid / LT, n - 1);
      const bf16_t* row = base + (long long)key * 3 * A + A + d;
      const long long at = (long long)min(key, positions - 1) * (D / 2) + d;
      kx[p] = *reinterpret_cast<const u32x4_v*>(row);
      ky[p] = *reinterpret_cast<const u32x4_v*>(row + D / 2);
      vx[p] = *reinterpret_cast<const u32x4_v*>(row + A);
      vy[p] = *reinterpret_cast<const u32x4_v*>(row + A + D / 2);
      ldv<float, 8>(cos_t + at, c[p]);
      ldv<float, 8>(sin_t + at, s[p]);
    }
  };
  fetch(0);
  // maxima are taken before the scale, which therefore has to be positive
  const bool negative = scale2 < 0.f;
  scale2 = fmaxf(fabsf(scale2), 1e-30f);
  bf16x8_v qf[KS];
  {
    u32x4_v qr[KS];
    const int t = min(w0 + col, n - 1);
    const bf16_t* row = base + (long long)t * 3 * A + hi * 8;
    const long long at = (long long)min(t, positions - 1) * (D / 2) + hi * 8;
#pragma unroll
    for (int k = 0; k < KS; ++k)
      qr[k] = *reinterpret_cast<const u32x4_v*>(row + k * 32);
#pragma unroll
    for (int k = 0; k < KS / 2; ++k) {
      float qc[8], qs[8];
      ldv<float, 8>(cos_t + at + k * 32, qc);
      ldv<float, 8>(sin_t + at + k * 32, qs);
      enc_rotate(qr[k], qr[k + KS / 2], qc, qs);
    }
#pragma unroll
    for (int k = 0; k < KS; ++k)
      qf[k] = __builtin_bit_cast(bf16x8_v,
                                 negative ? qr[k] ^ 0x80008000u : qr[k]);
  }
  f32x4_v acc[ET];
#pragma unroll
  for (int t = 0; t < ET; ++t) acc[t] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  float m = -3.0e38f, l = 0.f;
  const int tiles = (n + ENC_KEYS - 1) / ENC_KEYS;
  for (int tile = 0; tile < tiles; ++tile) {
    lds_barrier();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int key = p * TB + tid / LT;
      enc_rotate(kx[p], ky[p], c[p], s[p]);
      const bool ok = tile * ENC_KEYS + key < n;
      const u32x4_v zero = {0, 0, 0, 0};
      *reinterpret_cast<u32x4_v*>(&kt[key * KP + d]) = kx[p];
      *reinterpret_cast<u32x4_v*>(&kt[key * KP + d + D / 2]) = ky[p];
      *reinterpret_cast<u32x4_v*>(&vt[key * VP + d]) = ok ? vx[p] : zero;
      *reinterpret_cast<u32x4_v*>(&vt[key * VP + d + D / 2]) =
          ok ? vy[p] : zero;
    }
    lds_barrier();
    if (tile + 1 < tiles) fetch(tile + 1);
    if (w0 >= n) continue;             // nothing for this wave

    const int left = n - tile * ENC_KEYS;
    float alpha, top, psum;
    uint2 pk[4];
    // edge: some keys are hidden, 16 without one are left out; guard: a NaN score counts as no key
    auto weigh = [&](auto edge, auto guard) {
      f32x4_v sc[4];
      float mx = -INFINITY;
#pragma unroll
      for (int pt = 0; pt < 4; ++pt) {
        if (edge.value && pt * 16 >= left) break;
        sc[pt] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KS; ++k)
          sc[pt] = mfma_bf16(
              *reinterpret_cast<const bf16x8_v*>(
                  &kt[(pt * 16 + col) * KP + k * 32 + hi * 8]),
              qf[k], sc[pt]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (edge.value)
            if (pt * 16 + hi * 4 + r >= left) sc[pt][r] = -INFINITY;
          if constexpr (guard.value) sc[pt][r] = fmaxf(sc[pt][r], -INFINITY);
          mx = fmaxf(mx, sc[pt][r]);
        }
      }
      mx = rows_max(mx);
      top = fmaxf(m, mx * scale2);
      alpha = __builtin_amdgcn_exp2f(m - top);
      psum = 0.f;
#pragma unroll
      for (int pt = 0; pt < 4; ++pt) {
        if (edge.value && pt * 16 >= left) {
          pk[pt] = make_uint2(0, 0);
          continue;
        }
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[r] = __builtin_amdgcn_exp2f(fmaf(sc[pt][r], scale2, -top));
          psum += p[r];
        }
        pk[pt] = make_uint2(cvt_bf16x2(p[0], p[1]), cvt_bf16x2(p[2], p[3]));
      }
    };
    if (left >= ENC_KEYS) weigh(std::false_type{}, std::false_type{});
    else weigh(std::true_type{}, std::false_type{});
    // once more from LDS: kept scores would take registers from every tile
    if (__any(!(psum <= 64.f))) weigh(std::true_type{}, std::true_type{});
    m = top;
    l = l * alpha + psum;
#pragma unroll
    for (int t = 0; t < ET; ++t) acc[t] *= alpha;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k * 32 >= left) break;
      const bf16x8_v pf = __builtin_bit_cast(
          bf16x8_v, make_uint4(pk[2 * k].x, pk[2 * k].y, pk[2 * k + 1].x,
                               pk[2 * k + 1].y));
#pragma unroll
      for (int t = 0; t < ET; ++t)
        acc[t] = mfma_bf16(lds_frag_tr(vt, VP, k * 32, k * 32 + 16, t * 16,
                                       lane),
                           pf, acc[t]);
    }
  }
  l = rows_sum(l);
  const int t = w0 + col;
  if (t >= n) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  bf16_t* orow = out + (r0 + t) * A + (long long)h * D;
#pragma unroll
  for (int e = 0; e < ET; ++e) {
    const f32x4_v o = acc[e] * inv;
    *reinterpret_cast<uint2*>(orow + e * 16 + hi * 4) =
        make_uint2(cvt_bf16x2(o[0], o[1]), cvt_bf16x2(o[2], o[3]));
  }
}

extern "C" void qsa_encoder_attn_launch(
    const bf16_t* qkv, const float* cos_t, const float* sin_t, int positions,
    const int* qb_item, const int* qb_t0, const int* off, const int* len,
    bf16_t* out, int blocks, int H, int D, float scale, hipStream_t st) {
  if (blocks == 0) return;
  const dim3 grid((unsigned)((long long)blocks * H));
  const float scale2 = scale * 1.4426950408889634f;
  if (D == 128)
    hipLaunchKernelGGL(qsa_encoder_attn<128>, grid, dim3(256), 0, st, qkv,
                       cos_t, sin_t, positions, qb_item, qb_t0, off, len, out,
                       H, scale2);
  else
    hipLaunchKernelGGL(qsa_encoder_attn<64>, grid, dim3(256), 0, st, qkv,
                       cos_t, sin_t, positions, qb_item, qb_t0, off, len, out,
                       H, scale2);
}
