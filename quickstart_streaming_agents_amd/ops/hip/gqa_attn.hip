// Grouped-query attention over paged keys and values, with a per-head softmax
// sink and an output gate; key and value sizes are independent.
//
// Pages are row-major per key head: k [pages, G, 64, D], v [pages, G, 64, E],
// so a page of a key head is one contiguous tile for both sides, and a new
// token writes whole rows.  H / G query heads read the same tile.
//   out = softmax-with-sink(q.k * scale) v * sigmoid(gate) * out_scale
// The sink adds exp(sink_h) to the denominator: no key, no value, no scale.
//
//   qsa_gqa_rows        one block per (row, head), any size and storage type
//   qsa_gqa_rows_mfma   single rows and short portions: a wave takes a share
//                       of a row's pages for up to 16 heads of a key head
//                       (+ qsa_gqa_merge)
//   qsa_gqa_portions    flash attention of longer portions, page by page
#include <type_traits>

#include "lm_common.h"

#define PG 64
#define NEG_BIG (-3.0e38f)
#define LOG2E 1.4426950408889634f

// 2^x by the hardware instruction; what would be denormal becomes zero
__device__ __forceinline__ float exp2_hw(float x) {
  return __builtin_amdgcn_exp2f(x);
}

template <typename T>
__global__ void __launch_bounds__(256)
qsa_gqa_rows(const T* __restrict__ q, const T* __restrict__ kc,
             const T* __restrict__ vc, const int* __restrict__ block_table,
             int max_pages, const int* __restrict__ row_item,
             const int* __restrict__ row_len, const float* __restrict__ sink,
             const T* __restrict__ gate, long long gstride,
             T* __restrict__ out, long long ostride, int H, int G, int D,
             int E, float scale, float out_scale) {
  extern __shared__ float sm[];
  float* qs = sm;              // D
  float* os = qs + D;          // E
  __shared__ float sc[PG], ps[PG];
  const long long row = blockIdx.x / H;
  const int h = blockIdx.x % H, g = h / (H / G);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int k = tid; k < D; k += 256) qs[k] = ldf<T>(q + (row * H + h) * D + k);
  for (int k = tid; k < E; k += 256) os[k] = 0.f;
  int n = row_len[row];
  n = n > max_pages * PG ? max_pages * PG : n;
  const int* bt = block_table +
                  (long long)(row_item ? row_item[row] : row) * max_pages;
  float m = NEG_BIG, l = 0.f;
  __syncthreads();
  for (int pg = 0; pg * PG < n; ++pg) {
    const long long tile = ((long long)bt[pg] * G + g) * PG;
    const int b = min(n - pg * PG, PG);
    for (int j = wave; j < PG; j += 4) {
      float s = NEG_BIG;
      if (j < b) {
        s = 0.f;
        for (int k = lane; k < D; k += 64)
          s = fmaf(qs[k], ldf<T>(kc + (tile + j) * D + k), s);
        s = wave_reduce_sum(s) * scale;
      }
      if (lane == 0) sc[j] = s;
    }
    __syncthreads();
    const float mn = fmaxf(m, wave_reduce_max(sc[lane]));
    const float alpha = m > NEG_BIG ? expf(m - mn) : 0.f;
    const float p = sc[lane] > NEG_BIG ? expf(sc[lane] - mn) : 0.f;
    l = l * alpha + wave_reduce_sum(p);
    m = mn;
    if (wave == 0) ps[lane] = p;
    __syncthreads();
    for (int k = tid; k < E; k += 256) {
      float acc = os[k] * alpha;
      for (int j = 0; j < b; ++j)
        acc = fmaf(ps[j], ldf<T>(vc + (tile + j) * E + k), acc);
      os[k] = acc;
    }
  }
  const float sk = sink ? sink[h] : NEG_BIG;
  const float top = fmaxf(m, sk);
  const float f = m > NEG_BIG ? expf(m - top) : 0.f;
  const float den = l * f + (sink ? expf(sk - top) : 0.f);
  const float inv = den > 0.f ? f / den * out_scale : 0.f;
  for (int k = tid; k < E; k += 256) {
    float v = os[k] * inv;
    if (gate) v *= sigmoid_f(ldf<T>(gate + row * gstride + (long long)h * E + k));
    stf<T>(out + row * ostride + (long long)h * E + k, v);
  }
}

extern "C" void qsa_gqa_rows_launch(
    const void* q, const void* kc, const void* vc, const int* block_table,
    int max_pages, const int* row_item, const int* row_len, const float* sink,
    const void* gate, long long gstride, void* out, long long ostride, int R,
    int H, int G, int D, int E, float scale, float out_scale, int f32,
    hipStream_t st) {
  dim3 grid((unsigned)((long long)R * H));
  const size_t lds = sizeof(float) * ((size_t)D + E);
#define QSA_GR(T)                                                            \
  hipLaunchKernelGGL((qsa_gqa_rows<T>), grid, dim3(256), lds, st,            \
                     (const T*)q, (const T*)kc, (const T*)vc, block_table,   \
                     max_pages, row_item, row_len, sink, (const T*)gate,     \
                     gstride, (T*)out, ostride, H, G, D, E, scale, out_scale)
  if (f32) QSA_GR(float); else QSA_GR(bf16_t);
#undef QSA_GR
}

// ---------------------------------------------------------------------------
// Rows on the matrix cores.  Unit = (row, key head, 16 of its query heads,
// split of the pages), one WAVE each, no barriers: scores (A = keys straight
// from the page, B = queries in registers) leave softmax state and P^T
// lane-local (column = query head), V passes through the wave's own LDS tile
// for the transposing read.  A wave goes 32 positions at a time; the next
// keys are fetched once the scores are done, the next values once these are
// in LDS.  Bound by the read of the pages.
// MERGE: a block's four waves are the shares of one (row, key head, heads) and
// finish it in LDS; without, shares meet in qsa_gqa_merge (64 rows of 600-1400
// keys, 16 heads on 8 of 128: 68 + 6 us so, 69 us here, 3.9 TB/s).
// ---------------------------------------------------------------------------
struct GqaFinish {
  const float* sink;
  const bf16_t* gate;
  bf16_t* out;
  long long gstride, ostride;
  float out_scale;
};

// FAR: past the last-level cache.
template <int KS, int ET, bool MERGE, bool FAR>  // D <= 32*KS, E <= 16*ET
__device__ __forceinline__ void
gqa_rows(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
         const bf16_t* __restrict__ vc, const int* __restrict__ block_table,
         int max_pages, const int* __restrict__ row_item,
         const int* __restrict__ row_len, float* __restrict__ part_o,
         float* __restrict__ part_ml, int H, int G, int D, int E, float scale2,
         int NS, int units, const GqaFinish& fin,
         bf16_t (*vt_all)[32 * (16 * ET + 16)], float (*ml)[16][2]) {
  constexpr int VP = 16 * ET + 16;
  constexpr int VG = 2 * ET;                      // 16 B groups per V row
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int unit = blockIdx.x * 4 + wave;
  if (unit >= units) return;                      // MERGE: never
  bf16_t* vt = vt_all[wave];
  const int RG = H / G, HT = (RG + 15) / 16;
  const int split = unit % NS;
  const int ht = unit / NS % HT;
  const int g = unit / (NS * HT) % G;
  const long long row = unit / (NS * HT * G);
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, hi = lane >> 4;
  const int hg = ht * 16 + col;                   // head within the group
  const int head = g * RG + min(hg, RG - 1);
  const int n = min(row_len[row], max_pages * PG);
  const int np = n > 0 ? (n + PG - 1) / PG : 0;
  const int per = (np + NS - 1) / NS;
  const int ia = split * per * 2;                 // in steps of 32 positions
  const int ib = min((n + 31) / 32, ia + per * 2);
  const int* bt = block_table +
                  (long long)(row_item ? row_item[row] : row) * max_pages;
  float m = NEG_BIG, l = 0.f;
  f32x4_v acc[ET];
#pragma unroll
  for (int t = 0; t < ET; ++t) acc[t] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  if (n > 0 && ia < ib) {                         // uniform over the wave
    const bf16x8_v zero = {0, 0, 0, 0, 0, 0, 0, 0};
    bf16x8_v qf[KS], kf[2][KS];
    u32x4_v vr[ET];
    const bf16_t* qr = q + (row * H + head) * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int d = s * 32 + hi * 8;              // D % 8 == 0
      const bf16x8_v v = *reinterpret_cast<const bf16x8_v*>(
          qr + (d < D ? d : 0));
      qf[s] = d < D ? v : zero;
    }
    auto fetch_k = [&](int i) {
      const bf16_t* kb = kc + (((long long)bt[i >> 1] * G + g) * PG +
                               (i & 1) * 32) * D;
#pragma unroll
      for (int pt = 0; pt < 2; ++pt)
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const int d = s * 32 + hi * 8;          // past D: times zero
          const bf16x8_v* at = reinterpret_cast<const bf16x8_v*>(
              kb + (unsigned)((pt * 16 + col) * D + (d < D ? d : 0)));
          kf[pt][s] = FAR ? __builtin_nontemporal_load(at) : *at;
        }
    };
    auto fetch_v = [&](int i) {
      const bf16_t* vb = vc + (((long long)bt[i >> 1] * G + g) * PG +
                               (i & 1) * 32) * E;
#pragma unroll
      for (int u = 0; u < ET; ++u) {
        const int k = lane + u * 64;
        const int r = k / VG, c = (k % VG) * 8;
        const bool ok = c < E && i * 32 + r < n;
        const u32x4_v* at = reinterpret_cast<const u32x4_v*>(
            vb + (unsigned)(ok ? r * E + c : 0));
        const u32x4_v v = FAR ? __builtin_nontemporal_load(at) : *at;
        vr[u] = ok ? v : (u32x4_v){0, 0, 0, 0};
      }
    };
    fetch_k(ia);
    fetch_v(ia);
    for (int i = ia; i < ib; ++i) {
      f32x4_v s4[2];
#pragma unroll
      for (int pt = 0; pt < 2; ++pt) {
        f32x4_v a4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          bf16x8_v a = kf[pt][s];
          if (s * 32 + hi * 8 >= D) a = zero;
          a4 = mfma_bf16(a, qf[s], a4);
        }
        s4[pt] = a4;
      }
      if (i + 1 < ib) fetch_k(i + 1);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < ET; ++u) {
        const int k = lane + u * 64;
        *reinterpret_cast<u32x4_v*>(&vt[(k / VG) * VP + (k % VG) * 8]) = vr[u];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
      if (i + 1 < ib) fetch_v(i + 1);
      float mx = NEG_BIG;
#pragma unroll
      for (int pt = 0; pt < 2; ++pt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int p = i * 32 + pt * 16 + hi * 4 + r;
          s4[pt][r] = p < n ? s4[pt][r] * scale2 : NEG_BIG;
          mx = fmaxf(mx, s4[pt][r]);
        }
      mx = rows_max(mx);
      const float mn = fmaxf(m, mx);
      const float alpha = exp2_hw(m - mn);        // a step sees a key: mn is
                                                  // finite, masked terms 0
      m = mn;
      float psum = 0.f;
      uint2 pk[2];
#pragma unroll
      for (int pt = 0; pt < 2; ++pt) {
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[r] = exp2_hw(s4[pt][r] - mn);
          psum += p[r];
        }
        pk[pt] = make_uint2(cvt_bf16x2(p[0], p[1]), cvt_bf16x2(p[2], p[3]));
      }
      l = l * alpha + psum;
#pragma unroll
      for (int t = 0; t < ET; ++t) acc[t] *= alpha;
      const bf16x8_v pf = __builtin_bit_cast(
          bf16x8_v, make_uint4(pk[0].x, pk[0].y, pk[1].x, pk[1].y));
#pragma unroll
      for (int t = 0; t < ET; ++t)
        acc[t] = mfma_bf16(lds_frag_tr(vt, VP, 0, 16, t * 16, lane), pf,
                           acc[t]);
    }
    l = rows_sum(l);
  }
  if constexpr (MERGE) {
    // [16 heads][E] of every wave where its values were
    float* mine = reinterpret_cast<float*>(vt);
    __builtin_amdgcn_wave_barrier();
    if (hi == 0) {
      ml[wave][col][0] = m;
      ml[wave][col][1] = l;
    }
    if (n > 0 && ia < ib)
#pragma unroll
      for (int t = 0; t < ET; ++t)
        *reinterpret_cast<f32x4_v*>(mine + col * (16 * ET) + t * 16 + hi * 4) =
            acc[t];
    __syncthreads();
    const int heads = min(16, RG - ht * 16);
    for (int i = threadIdx.x; i < heads * (E / 2); i += 256) {
      const int hd = i / (E / 2), e = i % (E / 2) * 2;
      const int h = g * RG + ht * 16 + hd;
      const float sk = fin.sink ? fin.sink[h] * LOG2E : NEG_BIG;
      float top = sk;
#pragma unroll
      for (int w = 0; w < 4; ++w)
        if (ml[w][hd][1] > 0.f) top = fmaxf(top, ml[w][hd][0]);
      float den = fin.sink ? exp2_hw(sk - top) : 0.f, a0 = 0.f, a1 = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if (!(ml[w][hd][1] > 0.f)) continue;      // a share without keys
        const float f = exp2_hw(ml[w][hd][0] - top);
        den = fmaf(f, ml[w][hd][1], den);
        const float2 v = *reinterpret_cast<const float2*>(
            reinterpret_cast<const float*>(vt_all[w]) + hd * (16 * ET) + e);
        a0 = fmaf(f, v.x, a0);
        a1 = fmaf(f, v.y, a1);
      }
      const float inv = den > 0.f ? fin.out_scale / den : 0.f;
      a0 *= inv;
      a1 *= inv;
      if (fin.gate) {
        const float2 gv = bf16x2_to_f32x2(
            *reinterpret_cast<const unsigned int*>(
                fin.gate + row * fin.gstride + (long long)h * E + e));
        a0 /= 1.f + __expf(-gv.x);
        a1 /= 1.f + __expf(-gv.y);
      }
      *reinterpret_cast<unsigned int*>(fin.out + row * fin.ostride +
                                       (long long)h * E + e) =
          cvt_bf16x2(a0, a1);
    }
    return;
  }
  if (hg < RG) {
    const long long o = (row * H + head) * NS + split;
    if (hi == 0) {
      part_ml[o * 2] = m;
      part_ml[o * 2 + 1] = l;
    }
#pragma unroll
    for (int t = 0; t < ET; ++t) {
      const int e = t * 16 + hi * 4;
      if (e < E)                                  // E % 8 == 0
        *reinterpret_cast<f32x4_v*>(part_o + o * E + e) = acc[t];
    }
  }
}

// BOTH: past the cache if all rows together have more than far_keys.
template <int KS, int ET, bool MERGE, bool BOTH>
__global__ void __launch_bounds__(256, KS <= 4 && ET <= 8 ? 2 : 1)
qsa_gqa_rows_mfma(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                  const bf16_t* __restrict__ vc,
                  const int* __restrict__ block_table, int max_pages,
                  const int* __restrict__ row_item,
                  const int* __restrict__ row_len,
                  float* __restrict__ part_o, float* __restrict__ part_ml,
                  int H, int G, int D, int E, float scale2, int NS,
                  int units, GqaFinish fin, int rows, float far_keys) {
  __shared__ __attribute__((aligned(16))) bf16_t vt[4][32 * (16 * ET + 16)];
  __shared__ float ml[4][16][2];                  // MERGE
  bool past = false;
  if constexpr (BOTH) {
    // the row's length and first page are on their way meanwhile
    const int unit = __builtin_amdgcn_readfirstlane(
        min(blockIdx.x * 4 + (threadIdx.x >> 6), (unsigned)units - 1));
    const int row = unit / (NS * ((H / G + 15) / 16) * G);
    const int n = row_len[row], page = block_table[(long long)row * max_pages];
    past = wave_total(row_len, rows, [=](int k) {
             return (float)min(max(k, 0), max_pages * PG);
           }) > far_keys;
    asm volatile("" ::"s"(n), "s"(page));
  }
  if (past)
    gqa_rows<KS, ET, MERGE, true>(q, kc, vc, block_table, max_pages, row_item,
                                  row_len, part_o, part_ml, H, G, D, E, scale2,
                                  NS, units, fin, vt, ml);
  else
    gqa_rows<KS, ET, MERGE, false>(q, kc, vc, block_table, max_pages, row_item,
                                   row_len, part_o, part_ml, H, G, D, E, scale2,
                                   NS, units, fin, vt, ml);
}

// Splits -> normalized, gated output; the sink joins the denominator here.
// Statistics are in powers of two.  WPR waves merge one (row, head): one where
// there are few splits, four that share them otherwise.
template <int WPR>
__global__ void __launch_bounds__(256)
qsa_gqa_merge(const float* __restrict__ part_o,
              const float* __restrict__ part_ml,
              const float* __restrict__ sink, const bf16_t* __restrict__ gate,
              long long gstride, bf16_t* __restrict__ out, long long ostride,
              long long total, int H, int E, int NS, float out_scale) {
  __shared__ float2 red[WPR == 1 ? 1 : WPR][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = wave % WPR;
  const long long rh = (long long)blockIdx.x * (4 / WPR) + wave / WPR;
  if (rh >= total) return;                        // WPR 4: never
  const int h = (int)(rh % H), lane = threadIdx.x & 63;
  const long long row = rh / H;
  const float2* ml = reinterpret_cast<const float2*>(part_ml) + rh * NS;
  const float sk = sink ? sink[h] * LOG2E : NEG_BIG;
  float top = NEG_BIG;
  for (int s = lane; s < NS; s += 64)
    if (ml[s].y > 0.f) top = fmaxf(top, ml[s].x);
  top = fmaxf(wave_reduce_max(top), sk);
  float den = 0.f;
  for (int s = lane; s < NS; s += 64)
    if (ml[s].y > 0.f) den = fmaf(exp2_hw(ml[s].x - top), ml[s].y, den);
  den = wave_reduce_sum(den) + (sink ? exp2_hw(sk - top) : 0.f);
  const float inv = den > 0.f ? out_scale / den : 0.f;
  for (int e0 = 0; e0 < E; e0 += 128) {           // E % 8 == 0
    const int e = e0 + lane * 2;
    const bool in = e < E;
    const float* po = part_o + rh * NS * E + (in ? e : 0);
    float a0 = 0.f, a1 = 0.f;
    for (int s0 = 0; s0 < NS; s0 += 64) {
      const int n = min(64, NS - s0);
      float w = 0.f;
      if (lane < n && ml[s0 + lane].y > 0.f)
        w = exp2_hw(ml[s0 + lane].x - top);
#pragma unroll 8
      for (int s = sub; s < n; s += WPR) {
        const float ws = __shfl(w, s, QSA_WAVE);
        const float2 v = *reinterpret_cast<const float2*>(
            po + (long long)(s0 + s) * E);
        a0 = fmaf(ws, v.x, a0);
        a1 = fmaf(ws, v.y, a1);
      }
    }
    if (WPR > 1) {
      red[sub % WPR][lane] = make_float2(a0, a1);
      __syncthreads();
      if (sub == 0) {
#pragma unroll
        for (int k = 1; k < WPR; ++k) {
          a0 += red[k][lane].x;
          a1 += red[k][lane].y;
        }
      }
      __syncthreads();
    }
    if (sub == 0 && in) {
      a0 *= inv;
      a1 *= inv;
      if (gate) {
        const float2 gv = bf16x2_to_f32x2(
            *reinterpret_cast<const unsigned int*>(
                gate + row * gstride + (long long)h * E + e));
        a0 /= 1.f + __expf(-gv.x);
        a1 /= 1.f + __expf(-gv.y);
      }
      *reinterpret_cast<unsigned int*>(out + row * ostride + (long long)h * E +
                                       e) = cvt_bf16x2(a0, a1);
    }
  }
}

extern "C" void qsa_gqa_rows_mfma_launch(
    const bf16_t* q, const bf16_t* kc, const bf16_t* vc,
    const int* block_table, int max_pages, const int* row_item,
    const int* row_len, const float* sink, const bf16_t* gate,
    long long gstride, float* part_o, float* part_ml, bf16_t* out,
    long long ostride, int R, int H, int G, int D, int E, float scale,
    float out_scale, int NS, hipStream_t st) {
  const int units = R * G * ((H / G + 15) / 16) * NS;
  dim3 grid((unsigned)((units + 3) / 4));
  const float scale2 = scale * LOG2E;
  const GqaFinish fin{sink, gate, out, gstride, ostride, out_scale};
  // pages of many rows, read once a step beside those of other layers, would drive
  // each other out of the last-level cache (16 heads on 8 of 128, 64 rows of 600-1400
  // keys, 4 layers of 268 MB: 68.9 us with loads that stay there, 52.7 with others);
  // rows that share pages (portions' few tokens) read them from L2.  As in
  // paged_attn.hip the kernel sums up the keys where the table has room for so many.
  const bool far =
      (long long)R * max_pages * G * (D + E) * 2 * PG > QSA_FAR_PAGES && !row_item;
  const float far_keys = (float)(QSA_FAR_PAGES / (G * (D + E) * 2));
#define QSA_GM(K, V)                                                          \
  if (part_o && far) QSA_GM_AS(K, V, false, true);                            \
  else if (part_o) QSA_GM_AS(K, V, false, false);                             \
  else if (far) QSA_GM_AS(K, V, true, true);                                  \
  else QSA_GM_AS(K, V, true, false)
#define QSA_GM_AS(K, V, MERGE, FAR)                                           \
  hipLaunchKernelGGL((qsa_gqa_rows_mfma<K, V, MERGE, FAR>), grid, dim3(256),  \
                     0, st, q, kc, vc, block_table, max_pages, row_item,      \
                     row_len, part_o, part_ml, H, G, D, E, scale2, NS,        \
                     units, fin, R, far_keys)
#define QSA_GM_E(K)                                                           \
  if (E <= 32) { QSA_GM(K, 2); }                                              \
  else if (E <= 64) { QSA_GM(K, 4); }                                         \
  else if (E <= 128) { QSA_GM(K, 8); }                                        \
  else { QSA_GM(K, 16); }
  if (D <= 32) { QSA_GM_E(1); }
  else if (D <= 64) { QSA_GM_E(2); }
  else if (D <= 128) { QSA_GM_E(4); }
  else { QSA_GM_E(8); }
#undef QSA_GM_E
#undef QSA_GM
#undef QSA_GM_AS
  if (!part_o) return;
  const long long total = (long long)R * H;
  if (NS > 8)
    hipLaunchKernelGGL((qsa_gqa_merge<4>), dim3((unsigned)total), dim3(256),
                       0, st, part_o, part_ml, sink, gate, gstride, out,
                       ostride, total, H, E, NS, out_scale);
  else
    hipLaunchKernelGGL((qsa_gqa_merge<1>), dim3((unsigned)((total + 3) / 4)),
                       dim3(256), 0, st, part_o, part_ml, sink, gate, gstride,
                       out, ostride, total, H, E, NS, out_scale);
}

// ---------------------------------------------------------------------------
// Flash attention of portions.  Block = (64*QT query rows, head): wave w owns
// QT tiles of 16 rows, every page tile of K and V goes through LDS once per
// block and is read by all waves, each fragment used for QT tiles.  O^T stays
// in accumulators (row = value column, column = query row), so softmax state,
// rescale and P^T are lane-local.  Blocks walk the key heads first: with G a
// multiple of the 8 dies, one die's cache keeps one key head.
// Beside the matrix cores the softmax's vector work bounds it: the hidden keys
// are looked for on the last pages only, maxima are taken before the scale,
// which then joins the exponent in one fma, and the output is rescaled only
// where a maximum moved (4 x 1700 tokens, 16 heads on 8 of 128: 144 us without,
// 135 us here).
// ---------------------------------------------------------------------------
template <int KS, int ET, int QT>  // D <= 32*KS, E <= 16*ET
__global__ void __launch_bounds__(256, KS <= 4 && ET <= 8 ? 2 : 1)
qsa_gqa_portions(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                 const bf16_t* __restrict__ vc,
                 const int* __restrict__ block_table, int max_pages,
                 const float* __restrict__ sink,
                 const bf16_t* __restrict__ gate, long long gstride,
                 const int* __restrict__ qb_item,
                 const int* __restrict__ qb_t0, const int* __restrict__ off,
                 const int* __restrict__ start, const int* __restrict__ len,
                 bf16_t* __restrict__ out, long long ostride, int H, int G,
                 int D, int E, float scale2, float out_scale) {
  constexpr int KP = 32 * KS + 8;
  constexpr int VP = 16 * ET + 16;
  constexpr int KG = 4 * KS, VG = 2 * ET;         // 16 B groups per row
  constexpr int KL = 64 * KG / 256, VL = (64 * VG + 255) / 256;
  __shared__ __attribute__((aligned(16))) bf16_t kt[64 * KP];
  __shared__ __attribute__((aligned(16))) bf16_t vt[64 * VP];
  const int RG = H / G;
  const int g = blockIdx.x % G;
  const int h = g * RG + blockIdx.x / G % RG;
  const int qb = blockIdx.x / H;
  const int it = qb_item[qb], t0 = qb_t0[qb];
  const int n = len[it], p0 = start[it], r0 = off[it];
  const int* bt = block_table + (long long)it * max_pages;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  const int w0 = t0 + wave * 16 * QT;             // first row of this wave

  // maxima are taken before the scale, which therefore has to be positive
  const bool negative = scale2 < 0.f;
  scale2 = fmaxf(fabsf(scale2), 1e-30f);
  const bf16x8_v zero = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8_v qf[QT][KS];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    const long long qrow = r0 + min(w0 + u * 16 + col, n - 1);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int d = s * 32 + hi * 8;              // D % 8 == 0
      bf16x8_v v = *reinterpret_cast<const bf16x8_v*>(
          q + (qrow * H + h) * D + (d < D ? d : 0));
      if (negative) v ^= (short)0x8000;
      qf[u][s] = d < D ? v : zero;
    }
  }
  f32x4_v acc[QT][ET];
  float m[QT], l[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    m[u] = NEG_BIG;
    l[u] = 0.f;
#pragma unroll
    for (int t = 0; t < ET; ++t) acc[u][t] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  }
  const int last = p0 + min(t0 + 64 * QT, n) - 1; // last visible position
  const int wlast = p0 + w0 + 16 * QT - 1;        // ... of this wave

  uint4 kr[KL], vr[VL];
  auto fetch = [&](int pg) {
    const long long tile = ((long long)bt[pg] * G + g) * PG;
    const int have = last - pg * PG;              // rows 0..have are visible
#pragma unroll
    for (int u = 0; u < KL; ++u) {
      const int i = tid + u * 256;
      const int r = i / KG, c = (i % KG) * 8;
      const bool ok = r <= have && c < D;
      const uint4 v = *reinterpret_cast<const uint4*>(
          kc + (tile + (ok ? r : 0)) * D + (ok ? c : 0));
      kr[u] = ok ? v : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < VL; ++u) {
      const int i = tid + u * 256;
      const int r = i / VG, c = (i % VG) * 8;
      const bool ok = r <= have && r < PG && c < E;
      const uint4 v = *reinterpret_cast<const uint4*>(
          vc + (tile + (ok ? r : 0)) * E + (ok ? c : 0));
      vr[u] = ok ? v : make_uint4(0, 0, 0, 0);
    }
  };
  fetch(0);
  for (int pg = 0; pg * PG <= last; ++pg) {
    lds_barrier();
#pragma unroll
    for (int u = 0; u < KL; ++u) {
      const int i = tid + u * 256;
      *reinterpret_cast<uint4*>(&kt[(i / KG) * KP + (i % KG) * 8]) = kr[u];
    }
#pragma unroll
    for (int u = 0; u < VL; ++u) {
      const int i = tid + u * 256;
      if (i < 64 * VG)
        *reinterpret_cast<uint4*>(&vt[(i / VG) * VP + (i % VG) * 8]) = vr[u];
    }
    lds_barrier();
    if ((pg + 1) * PG <= last) fetch(pg + 1);
    if (pg * PG > wlast) continue;                // nothing for this wave
    f32x4_v s4[QT][4];
#pragma unroll
    for (int pt = 0; pt < 4; ++pt) {
#pragma unroll
      for (int u = 0; u < QT; ++u) s4[u][pt] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bf16x8_v a = *reinterpret_cast<const bf16x8_v*>(
            &kt[(pt * 16 + col) * KP + s * 32 + hi * 8]);
#pragma unroll
        for (int u = 0; u < QT; ++u)
          s4[u][pt] = mfma_bf16(a, qf[u][s], s4[u][pt]);
      }
    }
    bf16x8_v pf[QT][2];
    float alpha[QT];
    bool moved = false;
    auto softmax = [&](auto edge) {               // edge: some keys are hidden
#pragma unroll
      for (int u = 0; u < QT; ++u) {
        const int qpos = min(p0 + w0 + u * 16 + col, last);
        float mx = -INFINITY;
#pragma unroll
        for (int pt = 0; pt < 4; ++pt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if constexpr (edge.value)
              if (pg * PG + pt * 16 + hi * 4 + r > qpos)
                s4[u][pt][r] = -INFINITY;
            mx = fmaxf(mx, s4[u][pt][r]);
          }
        mx = rows_max(mx);
        const float mn = fmaxf(m[u], mx * scale2);
        moved |= mn > m[u];
        alpha[u] = exp2_hw(m[u] - mn);            // page 0 shows every row a
                                                  // key: mn is finite
        m[u] = mn;
        float psum = 0.f;
        uint2 pk[4];
#pragma unroll
        for (int pt = 0; pt < 4; ++pt) {
          float p[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            p[r] = exp2_hw(fmaf(s4[u][pt][r], scale2, -mn));
            psum += p[r];
          }
          pk[pt] = make_uint2(cvt_bf16x2(p[0], p[1]), cvt_bf16x2(p[2], p[3]));
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
          pf[u][s] = __builtin_bit_cast(
              bf16x8_v, make_uint4(pk[2 * s].x, pk[2 * s].y, pk[2 * s + 1].x,
                                   pk[2 * s + 1].y));
        l[u] = l[u] * alpha[u] + psum;
      }
    };
    if (pg * PG + PG - 1 > p0 + w0) softmax(std::true_type{});
    else softmax(std::false_type{});
    if (__any(moved)) {                           // else every factor is 1
#pragma unroll
      for (int u = 0; u < QT; ++u)
#pragma unroll
        for (int t = 0; t < ET; ++t) acc[u][t] *= alpha[u];
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < ET; ++t) {
        const bf16x8_v a =
            lds_frag_tr(vt, VP, s * 32, s * 32 + 16, t * 16, lane);
#pragma unroll
        for (int u = 0; u < QT; ++u)
          acc[u][t] = mfma_bf16(a, pf[u][s], acc[u][t]);
      }
  }
  const float sk = sink ? sink[h] * LOG2E : NEG_BIG;
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    l[u] = rows_sum(l[u]);
    const float top = fmaxf(m[u], sk);
    const float f = m[u] > NEG_BIG ? exp2f(m[u] - top) : 0.f;
    const float den = l[u] * f + (sink ? exp2f(sk - top) : 0.f);
    const float inv = den > 0.f ? f / den * out_scale : 0.f;
    const int i = w0 + u * 16 + col;
    if (i < n) {
      const bf16_t* gr = gate + (long long)(r0 + i) * gstride +
                         (long long)h * E;
      bf16_t* orow = out + (long long)(r0 + i) * ostride + (long long)h * E;
#pragma unroll
      for (int t = 0; t < ET; ++t) {
        const int e = t * 16 + hi * 4;
        if (e < E) {                              // E % 8 == 0
          float o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = acc[u][t][r] * inv;
          if (gate) {
            float gv[4];
            ldv<bf16_t, 4>(gr + e, gv);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] /= 1.f + __expf(-gv[r]);
          }
          stv<bf16_t, 4>(orow + e, o);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The same for heads beyond 64.  Pages go straight into LDS, both K and V stand
// twice, and a turn has one barrier: turn pg loads K of page pg + 2 and V of
// page pg, and multiplies what came a turn before.  The softmax of page pg runs
// beside the products of page pg - 1 with its values, a few exponents to each
// fragment of V; the scores of page pg + 1 follow.  Maxima cross the groups of a
// column by lane swaps.  A wave's first and last page stand outside of its loop:
// paths that meet behind the products keep the accumulators twice.
// us, one page after the other with two barriers / here (16 heads on 8, 4 x 2000
// tokens unless said; keys x values): 128 x 128 4 x 1700-2048 115 / 104, 1 x
// 8192 356 / 330, 16 x 1024 134 / 125, 100 + 200 27.6 / 24.9; 64 x 128 94.4 / 91.2;
// 16 heads on 4: 256 x 64 183 / 128, 256 x 128 205 / 151, 128 x 256 350 / 288,
// 256 x 256 407 / 344.  Heads of 64 and 32 have little to multiply and are bound
// by the exponents, with three blocks a CU above (63.5 us for 4 x 2000; 69 here).
// ---------------------------------------------------------------------------
template <int KS, int ET, int QT>  // D <= 32*KS, E <= 16*ET
__global__ void __launch_bounds__(256, ET <= 8 ? 2 : 1)
qsa_gqa_portions_beside(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                 const bf16_t* __restrict__ vc,
                 const int* __restrict__ block_table, int max_pages,
                 const float* __restrict__ sink,
                 const bf16_t* __restrict__ gate, long long gstride,
                 const int* __restrict__ qb_item,
                 const int* __restrict__ qb_t0, const int* __restrict__ off,
                 const int* __restrict__ start, const int* __restrict__ len,
                 bf16_t* __restrict__ out, long long ostride, int H, int G,
                 int D, int E, float scale2, float out_scale) {
#ifdef __HIP_DEVICE_COMPILE__          // loads into LDS: not for the host
  constexpr int KP = 32 * KS, VP = 16 * ET;       // elements of an LDS row
  constexpr int KG = KP / 8, VG = VP / 8;         // its pieces of 16 bytes
  constexpr int PD = 4;                // fragments of K or V in registers
  constexpr int VN = KS == 8 && ET == 8 ? 1 : 2;  // pages of V in LDS: two
                                                  // blocks fit a CU
  __shared__ __attribute__((aligned(16))) bf16_t kt[2 * PG * KP];
  __shared__ __attribute__((aligned(16))) bf16_t vt[VN * PG * VP];
  const int RG = H / G;
  const int g = blockIdx.x % G;
  const int h = g * RG + blockIdx.x / G % RG;
  const int qb = blockIdx.x / H;
  const int it = __builtin_amdgcn_readfirstlane(qb_item[qb]);
  const int t0 = __builtin_amdgcn_readfirstlane(qb_t0[qb]);
  const int n = __builtin_amdgcn_readfirstlane(len[it]);
  const int p0 = __builtin_amdgcn_readfirstlane(start[it]);
  const int r0 = off[it];
  const auto table = (const __attribute__((address_space(4))) int*)(
      block_table + (long long)it * max_pages);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  const int w0 = t0 + wave * 16 * QT;             // first row of this wave
  const int last = p0 + min(t0 + 64 * QT, n) - 1; // last visible position
  // pages of the block, those with keys for this wave, and those whose keys
  // all its rows see
  const int pages = (last + PG) / PG;
  const int mine = w0 >= n ? 0 : min(p0 + w0 + 16 * QT - 1, last) / PG + 1;
  const int whole = (p0 + w0 + 1) / PG;

  // A load fills 1 KB of LDS in the order of the lanes, so their addresses are
  // permuted: place j of row r has the row's piece j ^ sw(r), with which a read
  // of a fragment meets every bank once (two rows twice at KS = 8).  Columns from
  // D on and rows without a key are outside of the descriptor, which reads as
  // zero, and so do slots that nobody has written yet.
  auto ksw = [](int r) {
    return KS == 1 ? r >> 2 & 3 : KS == 2 ? r >> 1 & 7 : KS == 4 ? r & 15
                                                                 : r & 7;
  };
  auto vsw = [](int r) {
    return (ET == 2 ? r >> 2 & 1 : ET == 4 ? r >> 1 & 3 : r & 7) * 2;
  };
  const int kj = (lane % KG) ^ ksw((wave * 64 + lane) / KG);
  const int vj = (lane % VG) ^ vsw((wave * 64 + lane) / VG);
  const unsigned kfrom =
      kj * 8 < D ? (lane / KG) * D * 2 + kj * 16 : 0x7fffffffu;
  const unsigned vfrom =
      vj * 8 < E ? (lane / VG) * E * 2 + vj * 16 : 0x7fffffffu;
  auto load = [&](const bf16_t* cache, bf16_t* to, int pg, int place,
                  int width, unsigned from,
                  auto pieces) __attribute__((always_inline)) {
    constexpr int PR = decltype(pieces)::value;   // of a row
    const bf16_t* tile = cache + ((long long)table[pg] * G + g) * PG * width;
    const int bytes = min(last - pg * PG + 1, PG) * width * 2;
#pragma unroll
    for (int i = 0; i < PR / 4; ++i) {
      const int at = (wave + 4 * i) * (64 / PR) * width * 2;  // bytes before
      const __amdgpu_buffer_rsrc_t part = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(tile + at / 2), 0, max(bytes - at, 0), 0x00027000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          part, (__attribute__((address_space(3))) void*)(
                    to + place * PG * PR * 8 + (wave + 4 * i) * 512),
          16, from, 0, 0, 0);
    }
  };
  using KGt = std::integral_constant<int, KG>;
  using VGt = std::integral_constant<int, VG>;
  // all that the waves loaded has arrived, and they have read what they wanted
  auto arrived = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(7 << 4);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  load(kc, kt, 0, 0, D, kfrom, KGt{});
  if (pages > 1) load(kc, kt, 1, 1, D, kfrom, KGt{});

  // maxima are taken before the scale, which therefore has to be positive
  const bool negative = scale2 < 0.f;
  scale2 = fmaxf(fabsf(scale2), 1e-30f);
  const bf16x8_v zero = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8_v qf[QT][KS];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    const long long qrow = r0 + min(w0 + u * 16 + col, n - 1);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int d = s * 32 + hi * 8;              // D % 8 == 0
      bf16x8_v v = *reinterpret_cast<const bf16x8_v*>(
          q + (qrow * H + h) * D + (d < D ? d : 0));
      if (negative) v ^= (short)0x8000;
      qf[u][s] = d < D ? v : zero;
    }
  }
  f32x4_v acc[QT][ET], sc[QT][4];
  bf16x8_v pf[QT][2];
  float m[QT], l[QT], alpha[QT], psum[QT], top[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    m[u] = NEG_BIG;
    l[u] = 0.f;
    alpha[u] = 1.f;
#pragma unroll
    for (int t = 0; t < ET; ++t) acc[u][t] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  }
  bool moved = false;                  // a maximum, by the last softmax

  // fragment c of a page: keys of tile c % 4, k-step c / 4; values of rows
  // 32(c / ET).., columns 16(c % ET)..
  auto keys = [&](const bf16_t* k, int c) __attribute__((always_inline)) {
    const int r = (c & 3) * 16 + col;
    return *reinterpret_cast<const bf16x8_v*>(
        k + r * KP + (((c >> 2) * 4 + hi) ^ ksw(col)) * 8);
  };
  const int vr = hi * 4 + (col >> 2);
  auto vals = [&](const bf16_t* v, int c) __attribute__((always_inline)) {
    const int s = c / ET, t = c % ET;
    const bf16_t* at = v + (s * 32 + vr) * VP + ((t * 2) ^ vsw(vr)) * 8 +
                       (lane & 3) * 4;
    return __builtin_shufflevector(lds_read_tr(at), lds_read_tr(at + 16 * VP),
                                   0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto scores = [&](const bf16_t* k) __attribute__((always_inline)) {
    bf16x8_v f[PD];
#pragma unroll
    for (int c = 0; c < PD - 1; ++c) f[c] = keys(k, c);
#pragma unroll
    for (int c = 0; c < 4 * KS; ++c) {
      __builtin_amdgcn_sched_barrier(0);
      if (c + PD - 1 < 4 * KS) f[(c + PD - 1) % PD] = keys(k, c + PD - 1);
#pragma unroll
      for (int u = 0; u < QT; ++u)
        sc[u][c & 3] = mfma_bf16(
            f[c % PD], qf[u][c >> 2],
            c < 4 ? (f32x4_v){0.f, 0.f, 0.f, 0.f} : sc[u][c & 3]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto maximum = [&](int u) __attribute__((always_inline)) {
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[u][i >> 2][i & 3]);
    top[u] = fmaxf(m[u], rows_max(mx) * scale2);      // page 0 shows every row a
    moved |= top[u] > m[u];                       // key: it is finite
    alpha[u] = exp2_hw(m[u] - top[u]);
    psum[u] = 0.f;
  };
  unsigned int pk[QT][8];
  auto weights = [&](int u, int j) __attribute__((always_inline)) {
    const float a = exp2_hw(fmaf(sc[u][j >> 1][(j & 1) * 2], scale2, -top[u]));
    const float b =
        exp2_hw(fmaf(sc[u][j >> 1][(j & 1) * 2 + 1], scale2, -top[u]));
    psum[u] += a;
    psum[u] += b;
    pk[u][j] = cvt_bf16x2(a, b);
  };
  auto packed = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < QT; ++u) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
        pf[u][s] = __builtin_bit_cast(
            bf16x8_v, make_uint4(pk[u][4 * s], pk[u][4 * s + 1],
                                 pk[u][4 * s + 2], pk[u][4 * s + 3]));
      m[u] = top[u];
      l[u] = l[u] * alpha[u] + psum[u];
    }
  };
  // softmax of sc by itself
  auto first = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      maximum(u);
#pragma unroll
      for (int j = 0; j < 8; ++j) weights(u, j);
    }
    packed();
  };
  auto products = [&](const bf16_t* v) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2 * ET; ++c) {
      const bf16x8_v a = vals(v, c);
#pragma unroll
      for (int u = 0; u < QT; ++u)
        acc[u][c % ET] = mfma_bf16(a, pf[u][c / ET], acc[u][c % ET]);
      if (c & 1) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // softmax of sc beside the products of the weights before it with v
  auto beside = [&](const bf16_t* v) __attribute__((always_inline)) {
    constexpr int NC = ET * 2, PAIRS = QT * 8, SPAN = NC - 2;
    bf16x8_v f[PD];
#pragma unroll
    for (int c = 0; c < PD - 1; ++c) f[c] = vals(v, c);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      __builtin_amdgcn_sched_barrier(0);
      if (c + PD - 1 < NC) f[(c + PD - 1) % PD] = vals(v, c + PD - 1);
#pragma unroll
      for (int u = 0; u < QT; ++u)
        acc[u][c % ET] = mfma_bf16(f[c % PD], pf[u][c / ET], acc[u][c % ET]);
      if (c < QT) maximum(c);
#pragma unroll
      for (int i = 0; i < PAIRS; ++i)
        if (c == 2 + i * SPAN / PAIRS) weights(i >> 3, i & 7);
    }
    __builtin_amdgcn_sched_barrier(0);
    packed();
  };

  arrived();
  if (mine > 0) scores(kt);
  // a turn's barrier and loads: K of page pg + 1 and V of pg - 1 are there
  auto stage = [&](int pg) __attribute__((always_inline)) {
    arrived();
    if (pg + 2 < pages) load(kc, kt, pg + 2, pg & 1, D, kfrom, KGt{});
    if (VN == 2 && pg < pages) load(vc, vt, pg, pg & 1, E, vfrom, VGt{});
  };
  // after a turn's products with values
  auto after = [&](int pg) __attribute__((always_inline)) {
    if constexpr (VN == 1) {
      lds_barrier();
      if (pg < pages) load(vc, vt, pg, 0, E, vfrom, VGt{});
    }
  };
  // keys of page pg that a row does not see
  auto hide = [&](int pg) __attribute__((always_inline)) {
    if (pg < whole) return;
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      const int see =
          min(p0 + w0 + u * 16 + col, last) - pg * PG - hi * 4;
#pragma unroll
      for (int pt = 0; pt < 4; ++pt) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (pt * 16 + r > see) sc[u][pt][r] = -INFINITY;
        __builtin_amdgcn_sched_barrier(0);  // few masks at a time
      }
    }
  };
  auto rescale = [&]() __attribute__((always_inline)) {
    if (__any(moved)) {                // else every factor is 1
#pragma unroll
      for (int u = 0; u < QT; ++u)
#pragma unroll
        for (int t = 0; t < ET; ++t) acc[u][t] *= alpha[u];
    }
    moved = false;
  };
  stage(0);
  after(0);
  int pg = 1;
  if (mine > 0) {
    hide(0);
    first();
    moved = false;                     // nothing to rescale
    if (mine > 1) scores(kt + PG * KP);
#pragma clang loop unroll(disable)
    for (; pg < mine; ++pg) {
      stage(pg);
      rescale();
      hide(pg);
      beside(vt + (VN == 2 ? (pg + 1) & 1 : 0) * PG * VP);
      after(pg);
      if (pg + 1 < mine) scores(kt + ((pg + 1) & 1) * PG * KP);
    }
    stage(pg);
    rescale();
    products(vt + (VN == 2 ? (pg + 1) & 1 : 0) * PG * VP);
    after(pg);
    ++pg;
  }
#pragma clang loop unroll(disable)
  for (; pg <= pages; ++pg) {
    stage(pg);
    after(pg);
  }
  const float sk = sink ? sink[h] * LOG2E : NEG_BIG;
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    l[u] = rows_sum(l[u]);
    const float top = fmaxf(m[u], sk);
    const float f = m[u] > NEG_BIG ? exp2f(m[u] - top) : 0.f;
    const float den = l[u] * f + (sink ? exp2f(sk - top) : 0.f);
    const float inv = den > 0.f ? f / den * out_scale : 0.f;
    const int i = w0 + u * 16 + col;
    if (i < n) {
      const bf16_t* gr = gate + (long long)(r0 + i) * gstride +
                         (long long)h * E;
      bf16_t* orow = out + (long long)(r0 + i) * ostride + (long long)h * E;
#pragma unroll
      for (int t = 0; t < ET; ++t) {
        const int e = t * 16 + hi * 4;
        if (e < E) {                              // E % 8 == 0
          float o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = acc[u][t][r] * inv;
          if (gate) {
            float gv[4];
            ldv<bf16_t, 4>(gr + e, gv);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] /= 1.f + __expf(-gv[r]);
          }
          stv<bf16_t, 4>(orow + e, o);
        }
      }
    }
  }
#endif
}

extern "C" void qsa_gqa_portions_launch(
    const bf16_t* q, const bf16_t* kc, const bf16_t* vc,
    const int* block_table, int max_pages, const float* sink,
    const bf16_t* gate, long long gstride, const int* qb_item,
    const int* qb_t0, const int* off, const int* start, const int* len,
    bf16_t* out, long long ostride, int QB, int H, int G, int D, int E,
    float scale, float out_scale, int wide, hipStream_t st) {
  dim3 grid((unsigned)((long long)QB * H));
  const float scale2 = scale * LOG2E;
#define QSA_GP(K, V, Q)                                                      \
  if constexpr (K <= 2 && V <= 4) QSA_GP_AS(qsa_gqa_portions, K, V, Q);      \
  else QSA_GP_AS(qsa_gqa_portions_beside, K, V, Q)
#define QSA_GP_AS(NAME, K, V, Q)                                             \
  hipLaunchKernelGGL((NAME<K, V, Q>), grid, dim3(256), 0, st, q,             \
                     kc, vc, block_table, max_pages, sink, gate, gstride,    \
                     qb_item, qb_t0, off, start, len, out, ostride, H, G, D, \
                     E, scale2, out_scale)
#define QSA_GP_E(K, W)                                                       \
  if (E <= 32) { if (W) QSA_GP(K, 2, 2); else QSA_GP(K, 2, 1); }             \
  else if (E <= 64) { if (W) QSA_GP(K, 4, 2); else QSA_GP(K, 4, 1); }        \
  else if (E <= 128) { if (W) QSA_GP(K, 8, 2); else QSA_GP(K, 8, 1); }       \
  else QSA_GP(K, 16, 1)
  if (D <= 32) { QSA_GP_E(1, wide); }
  else if (D <= 64) { QSA_GP_E(2, wide); }
  else if (D <= 128) { QSA_GP_E(4, wide); }
  else if (E <= 128) { if (E <= 32) QSA_GP(8, 2, 1);
                       else if (E <= 64) QSA_GP(8, 4, 1);
                       else QSA_GP(8, 8, 1); }
  else { QSA_GP(8, 16, 1); }
#undef QSA_GP_E
#undef QSA_GP
#undef QSA_GP_AS
}
