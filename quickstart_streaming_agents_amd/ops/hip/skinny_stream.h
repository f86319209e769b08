// Weight-streaming decode GEMM for CDNA4 (gfx950), shared by the bf16 and the
// fp8 form: C[M,N] = A[M,K] @ W[N,K]^T for M <= 32 rows.
//
// The projections of a decoding step read every weight once, so the weight
// stream is the bound and the rest has to stay out of its way:
//   * W is packed once into MFMA fragments (layouts in skinny_gemm.hip and
//     skinny_gemm_fp8.hip): a wave instruction reads 1 KiB in a row.
//   * A block owns TILES tiles of 16 columns; its waves take the 64-deep steps
//     of K in turn, so that the block reads its stream front to back, and keep
//     two groups of U steps in flight.  They meet in LDS at the end.
//   * A is tiny and L2 holds it, but a row-major fragment touches 16 lines
//     where W's takes 8, and at 16 rows those lookups, not the weights, set
//     the pace (a tile per block: 28672 x 4096 fp8 in 25 us at 1 row, 38 us at
//     16).  From 5 rows on the decoder keeps its activations packed in
//     fragments like W (PACK: [K/32, MT, 64 lanes, 8]); producers store them
//     so.  MT row tiles of 16: one for up to 16 rows, two above.
//   * Row-major rows beyond M shadow row M-1, packed ones are whatever the
//     buffer holds; they meet no other row and are never stored.  Of a tile of
//     up to 8 rows the lanes of the others take the same lines: a block reads all
//     of A, twice the bytes of its weights at 16 rows (8 layers of width 4096, a step
//     of 8 rows 637 -> 560 us, of 6 554 -> 493, of 20 716 -> 686).
//   * FAR: where the weights of a step exceed the last-level cache, each of them
//     is driven out before the next step, and with it what would stay: keys and
//     values of small batches, activations, weights read ahead.  Their loads leave
//     no trace then (16 layers of width 2048, 1 row of 700 keys 577 -> 537 us a
//     step; 8 layers, 4 rows 357 -> 320; of width 4096, 1 row 547 -> 504).  Weights
//     that fit are to stay (8 layers of width 1024, 119 MB, 1 row: 187 us, 195 past
//     the cache).
// What surrounds a projection in the decoder is done on the way, since every
// launch costs a few microseconds of a step that is made of hundreds:
//   NORM  A is x * w of an rms norm; the row factor 1/rms meets the sums at the
//         end.  The sum of squares of a row comes in parts from whoever wrote
//         the row (ss_in [32, parts4], parts4 = parts rounded up to 4).
//   GLU   W's rows are [gate; up]: a block takes the same columns of both and
//         stores silu(gate) * up, packed if A is.
//   RES   the result is added to the residual stream in place; the next norm's
//         operand (new row * norm_w, packed if A is) goes to `next`, the
//         sums of squares of the new rows to ss_out, one part per tile.
//   HALF  a block has half a tile, for few columns, whose tiles would leave CUs idle
//         and the others a stream each that one memory latency does not cover.  Lanes
//         of columns 8 to 15 take the same eight columns further on in K, and rows 8
//         to 15 of A are its rows 0 to 7 there; the result is the sum of the two
//         diagonal quarters, so up to 8 rows.  One part of a sum per half.
// (Multiplying by w on the way in instead cost 20 us of 25 at 28672 x 4096:
// every block redoes it, and its loads take the place of the stream's.)
#pragma once

#include "lm_common.h"

struct SkinnyArgs {
  const bf16_t* A;
  const u32x4_v* W;
  const float* scale;                  // fp8: per output column
  bf16_t* C;                           // result, or the residual stream
  bf16_t* next;
  const bf16_t* norm_w;
  const float* ss_in;
  float* ss_out;
  int M, N, parts;
  long long K, lda;
  float eps;
  bool far;                            // W is read past the last-level cache
};

// 8 fp8 bytes (as 2 dwords) -> bf16x8 fragment, exact: every e4m3 value is a
// bf16 value, and the scale is one.  One conversion a pair: by way of f32 and a
// permutation it was twice the instructions (us a step, 16 layers of width 2048, one
// row 492 -> 486, 24 rows 741 -> 737; 8 layers of 4096, 16 rows 688 -> 682).
__device__ __forceinline__ bf16x8_v fp8x8_to_bf16x8(unsigned int a,
                                                    unsigned int b) {
  const u32x4_v u = {
      __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, false)),
      __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, true)),
      __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, false)),
      __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, true))};
  return __builtin_bit_cast(bf16x8_v, u);
}

// place of element k of a row in packed activations
__device__ __forceinline__ long long packed_at(int row, int k, int mt) {
  return ((long long)(k >> 5) * mt + (row >> 4)) * 512 +
         ((row & 15) + ((k >> 3) & 3) * 16) * 8 + (k & 7);
}

// How A is given: rows, fragments, or up to FEW rows.  Fragments of few rows are mostly
// lanes of rows that do not exist, and a load brings 1 KB into registers all the same,
// two of them for each of W: a wave loads the rows that are there, 128 bytes of each for
// a step, and lays them out in LDS (us a step: 8 layers of width 2048, 4 rows 269 -> 258;
// 16 layers, 3 rows 501 -> 484; one row level).
enum { ROWS = 0, PACKED = 1, FEW_ROWS = 2 };
#define FEW 4

template <int WAVES, int TILES, int MT, bool FP8, int FORM, bool NORM,
          bool GLU, bool RES, bool FAR, bool HALF = false>
__device__ __forceinline__ void skinny_stream(const SkinnyArgs& p) {
  static_assert(!HALF || (FP8 && RES && TILES == 1 && MT == 1), "half a tile");
  static_assert(FORM != FEW_ROWS || MT == 1, "few rows are one tile");
  constexpr bool PACK = FORM == PACKED, LITTLE = FORM == FEW_ROWS;
  constexpr int WL = FP8 ? 1 : 2;      // 16 B loads of a tile per step
  constexpr int PER = TILES * WL * 4 + MT * 8;
  constexpr int U = PER <= 12 ? 4 : PER <= 24 ? 2 : 1;
  // LITTLE: a wave's part of A for a group: rows of U steps of 128 bytes, 64 apart
  // in the banks; of half a tile both parts of K
  constexpr int LR = U * 64 + 32, LH = FEW * LR;  // elements of a row, of a part
  constexpr int AREA = LITTLE ? (HALF ? 2 : 1) * LH : 0;
  constexpr int AL = LITTLE ? (HALF ? 2 : 1) * FEW * U * 8 / 64 : 1;
  __shared__ __attribute__((aligned(16))) bf16_t few[WAVES * AREA + 8];
  __shared__ float red[WAVES][TILES * MT * 4][64];
  __shared__ float inv_s[32];
  const int tid = threadIdx.x, lane = tid & 63;
  // the wave's number as a scalar: branches on it must skip MFMAs, which
  // would otherwise run with no lane enabled and still add up
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  // K % 64 == 0, HALF: % 128 and steps of either half of K; A's offsets fit 31 bits
  const int steps = (int)(p.K >> (HALF ? 7 : 6));
  // a lane's column of its tile, as results are stored
  const int tcol = HALF ? ((int)blockIdx.x & 1) * 8 + (col & 7) : col;

  // row factors: the parts' loads go ahead of the stream, a row per wave
  constexpr int NR = NORM ? MT * 16 / WAVES : 1;
  f32x4_v sv[NR];
  const int p4 = (p.parts + 3) & ~3;
  if constexpr (NORM)
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int row = wave + i * WAVES;
      sv[i] = *reinterpret_cast<const f32x4_v*>(
          p.ss_in + (row < p.M ? row : 0) * p4 + (lane * 4 < p4 ? lane * 4 : 0));
    }

  // GLU: tiles 2j and 2j+1 are gate and up of the same 16 columns
  auto tile_of = [&](int t) {
    return GLU ? (int)blockIdx.x * (TILES / 2) + t / 2 +
                     (t & 1) * (p.N >> 5)
               : HALF ? (int)blockIdx.x >> 1 : (int)blockIdx.x * TILES + t;
  };
  // what the results need besides the sums is fetched ahead of the stream: at
  // the end each of these would be a memory latency of its own (2048 x 2048
  // fp8, 1 row: 4.5 -> 4.1 us; 4096 x 14336: 15.0 -> 14.3)
  constexpr int OUT = (GLU ? TILES / 2 : TILES) * MT * 256;
  constexpr int NI = (OUT + WAVES * 64 - 1) / (WAVES * 64);
  float sc[NI][GLU ? 2 : 1];
  bf16_t old[NI], nw[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int idx = min(tid + i * WAVES * 64, OUT - 1);
    const int r = (idx >> 6) & 3, m = (idx >> 8) % MT, j = (idx >> 8) / MT;
    if constexpr (FP8)
#pragma unroll
      for (int e = 0; e < (GLU ? 2 : 1); ++e)
        sc[i][e] = p.scale[tile_of(GLU ? 2 * j + e : j) * 16 + tcol];
    if constexpr (RES) {
      const int row = m * 16 + hi * 4 + r, c = tile_of(j) * 16 + tcol;
      old[i] = p.C[(long long)(row < p.M ? row : 0) * p.N + c];
      nw[i] = p.norm_w[c];
    }
  }
  // Where loads are: a tile's stream and A, a lane's place in them, and the step, which
  // is a scalar: no vector instruction makes an address.  Steps beyond the end are read
  // as zeros, from nowhere, and multiplied like others, so that a wave's code is short
  // and without branches; the groups are worked on as they arrive.  (us a step with
  // 64-bit addresses and a look at every step, and so: 16 layers of width 2048, one row
  // 485 -> 460, 24 rows 734 -> 705; 8 layers of 4096, one row 478 -> 467, 6 rows 514 ->
  // 502, 16 rows 680 -> 672.)
  using rsrc = __amdgpu_buffer_rsrc_t;
  constexpr int WB = 1024 * WL;                   // bytes of a tile's step
  const int stream = (HALF ? 2 : 1) * steps * WB;
  const unsigned wo = (unsigned)(tcol * 4 + hi) * 16 +
                      (HALF ? (unsigned)(col >> 3) * steps * WB : 0u);
  unsigned ao[LITTLE ? AL : MT];
  int am[AL], lo[AL];                             // LITTLE: steps ahead; place in LDS
  if constexpr (LITTLE) {
#pragma unroll
    for (int j = 0; j < AL; ++j) {
      const int i = j * 64 + lane, seg = i & 7, u = i / 8 % U;
      const int m = i / (8 * U) % FEW, h = i / (8 * U * FEW);
      am[j] = m < p.M ? u * WAVES : 0x40000000;
      ao[j] = ((unsigned)m * (unsigned)p.lda + (unsigned)(u * WAVES * 64 + seg * 8) +
               (unsigned)h * steps * 64) * 2;
      lo[j] = wave * AREA + h * LH + m * LR + u * 64 + seg * 8;
    }
  }
#pragma unroll
  for (int m = 0; m < (LITTLE ? 0 : MT); ++m)
    if constexpr (HALF)
      ao[m] = ((unsigned)(col >> 3) * steps * (PACK ? 1024 : 64) +
               (PACK ? ((col & 7) + hi * 16) * 8
                     : min(col & 7, p.M - 1) * (unsigned)p.lda + hi * 8)) * 2;
    else
      // packed rows that do not exist: the line of eight that do
      ao[m] = (PACK ? m * 512 + ((p.M - m * 16 <= 8 ? col & 7 : col) + hi * 16) * 8
                    : min(m * 16 + col, p.M - 1) * (unsigned)p.lda + hi * 8) * 2;

  struct Group {
    u32x4_v w[U][TILES][WL];
    bf16x8_v a[LITTLE ? 1 : U][MT][2];
    u32x4_v few[AL];
  };
  f32x4_v acc[TILES][MT];
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = (f32x4_v){0.f, 0.f, 0.f, 0.f};

  const rsrc rf = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, 0x7fffffff,
                                                    0x00027000);
  // from nowhere: just beyond what a descriptor covers, whatever the step adds to it
  constexpr unsigned NOWHERE = 0x80000000u;
  auto load = [&](Group& g, int base) {
    if constexpr (LITTLE)
#pragma unroll
      for (int j = 0; j < AL; ++j)
        g.few[j] = __builtin_amdgcn_raw_buffer_load_b128(
              rf, base + am[j] < steps ? ao[j] : NOWHERE, base * 128, 0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = base + u * WAVES;
      const bool in = s < steps;                  // uniform over the wave
      const int at = in ? s : 0;
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        const rsrc rw = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(p.W + (long long)tile_of(t) * (stream / 16)), 0,
            in ? stream : 0, 0x00027000);
#pragma unroll
        for (int i = 0; i < WL; ++i)
          g.w[u][t][i] = __builtin_amdgcn_raw_buffer_load_b128(
              rw, wo + i * 1024, at * WB, FAR ? QSA_NT : 0);
      }
      if constexpr (LITTLE) continue;
      const rsrc ra = __builtin_amdgcn_make_buffer_rsrc(
          (void*)p.A, 0, in ? 0x7fffffff : 0, 0x00027000);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          g.a[u][m][i] = __builtin_bit_cast(
              bf16x8_v, __builtin_amdgcn_raw_buffer_load_b128(
                            ra, ao[m] + i * (PACK ? MT * 1024 : 64),
                            at * (PACK ? MT * 2048 : 128), 0));
    }
  };
  const bf16_t* const fa =
      few + wave * AREA +
      (HALF ? (col >> 3) * LH + min(col & 7, p.M - 1) * LR
            : min(col, p.M - 1) * LR) + hi * 8;
  auto compute = [&](Group& g) {
    bf16x8_v f[U][2];
    if constexpr (LITTLE) {            // a wave's own: its order suffices
#pragma unroll
      for (int j = 0; j < AL; ++j)
        *reinterpret_cast<u32x4_v*>(few + lo[j]) = g.few[j];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          f[u][i] = *reinterpret_cast<const bf16x8_v*>(fa + u * 64 + i * 32);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          bf16x8_v w;
          if constexpr (FP8)
            w = fp8x8_to_bf16x8(g.w[u][t][0][2 * i], g.w[u][t][0][2 * i + 1]);
          else
            w = __builtin_bit_cast(bf16x8_v, g.w[u][t][i]);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[t][m] = mfma_bf16(LITTLE ? f[u][i] : g.a[LITTLE ? 0 : u][m][i], w,
                                  acc[t][m]);
        }
  };

  Group g0, g1;
  constexpr int ROUND = WAVES * U;
  load(g0, wave);
  load(g1, wave + ROUND);
  if constexpr (NORM) {
    auto factor = [&](int i) {
      const int row = wave + i * WAVES;
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) s += lane * 4 + e < p.parts ? sv[i][e] : 0.f;
      for (int k = 256 + lane; k < p.parts; k += 64)
        s += p.ss_in[row * p4 + k];
      s = wave_reduce_sum(s);
      if (lane == 0) inv_s[row] = rsqrtf(s / (float)p.K + p.eps);
    };
    // Rows that do not exist cost a wave 86 instructions each before its first
    // product (16 layers of width 2048, a step of one row 509 -> 494 us; 8 layers, 4
    // rows 293 -> 281).  Where all 16 do, the chains of a wave's rows lie beside each
    // other, without a look at each (us, looks / none: 16 rows of 2048 x 2048 3.93 /
    // 3.61, of 1024 x 768 3.79 / 3.58, of 512 x 256 3.72 / 3.56, 28,672 x 4096 gated
    // 23.7 / 23.3; of two tiles 32 rows of 16,384 x 2048 gated 7.9 / 8.3).
    if (MT == 1 && p.M == 16) {
#pragma unroll
      for (int i = 0; i < NR; ++i) factor(i);
    } else {
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        if (wave + i * WAVES >= p.M) break;       // uniform over the wave
        factor(i);
      }
    }
  }
  // both groups are always loaded again, so that the waits in the loop are for one
  for (int base = wave; base + 2 * ROUND < steps; base += 2 * ROUND) {
    compute(g0);
    load(g0, base + 2 * ROUND);
    compute(g1);
    load(g1, base + 3 * ROUND);
  }
  compute(g0);
  compute(g1);

#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wave][(t * MT + m) * 4 + r][lane] = acc[t][m][r];
  __syncthreads();

#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int idx = tid + i * WAVES * 64;
    if (OUT % (WAVES * 64) != 0 && idx >= OUT) break;
    const int r = (idx >> 6) & 3, m = (idx >> 8) % MT, j = (idx >> 8) / MT;
    const int row = m * 16 + (lane >> 4) * 4 + r;
    auto total = [&](int t, int e) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v += red[w][(t * MT + m) * 4 + r][lane];
      if constexpr (HALF)              // row + 8, column + 8
#pragma unroll
        for (int w = 0; w < WAVES; ++w) v += red[w][r][(lane + 40) & 63];
      if constexpr (FP8) v *= sc[i][e];
      return v;
    };
    const float inv = NORM ? inv_s[row] : 1.f;
    const int ncol = tile_of(GLU ? 2 * j : j) * 16 + tcol;
    const bool live = row < p.M && (!HALF || (row < 8 && col < 8));
    auto place = [&](int width) {
      return PACK ? packed_at(row, ncol, MT) : (long long)row * width + ncol;
    };
    if constexpr (GLU) {
      const float g = total(2 * j, 0) * inv, u = total(2 * j + 1, GLU) * inv;
      if (live)
        p.C[place(p.N >> 1)] = cvt_bf16(g / (1.f + __expf(-g)) * u);
    } else if constexpr (RES) {
      const float v = bf16_to_f32(old[i]) + total(j, 0);
      const bf16_t b = cvt_bf16(v);
      if (live) {
        p.C[(long long)row * p.N + ncol] = b;
        p.next[place(p.N)] = cvt_bf16(bf16_to_f32(b) *
                                      bf16_to_f32(nw[i]));
      }
      const float q = row16_sum(HALF && col >= 8 ? 0.f : v * v);
      constexpr int PART = HALF ? 3 : 4;           // log2 of its columns
      const int parts = p.N >> PART;
      if (live && col == 0)
        p.ss_out[row * ((parts + 3) & ~3) + (ncol >> PART)] = q;
    } else {
      const float v = total(j, 0) * inv;
      if (live) p.C[(long long)row * p.N + ncol] = cvt_bf16(v);
    }
  }
}
