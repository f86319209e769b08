// GEMM of many rows: C[M,N] = A[M,K] @ W[N,K]^T, bf16 with f32 sums, or
// act(gate) * up of it with W = [gate; up], where the largest tiles fill the chip.
//
// What bounds it is power, and before that the way from L2 into LDS: a stage of
// 256 x 256 (64 KB for 2048 cycles of products) arrives some 1.5 us after its loads
// where all CUs load at once, and with two stages in LDS they are asked for one stage
// ahead, 1.1 us.  Hence places for A of two stages and for W of three (160 KB in all):
// W's loads go out half a stage earlier and A's have the way to themselves.  Cycles a
// stage 2900 -> 2450 (2170 without loads), and the clock falls from 1.93 to 1.75 GHz.
// Four waves of 128 x 128 read a third less from LDS than eight of 128 x 64 (with both
// operands two stages deep they are slower, 3200 cycles).  Blocks stay for all their
// tiles: the next one's first two stages are under way while a tile is stored, from
// registers, for W's rows lie in LDS so that a lane's results are eight neighbours.
// Every product shares an operand with the one before, which is 2 % (less switches).
// PFLOP/s of random data, the library's -> here (the 8-wave tile of rows_gemm.hip):
//   8192 x 8192 x 4096    1.61 -> 1.59 (1.47)     8192 x 28672 x 4096  1.58 -> 1.54 (1.37)
//   44800 x 4096 x 14336  1.43 -> 1.50 (1.32)     10816 x 4096 x 4096  0.93 -> 1.40 (1.33)
// us, the activation a pass of its own beside the library's product:
//   rows           512          2048         7500          13800         44800
//   6144 x 4096    30.8 -> 27.5  78.3 -> 72.0  252 -> 256    549 -> 480    1581 -> 1516
//   4096 x 14336   76 -> (63)    187 -> 172    998 -> 614    1254 -> 1179  3719 -> 3568
//   28672 x 4096 (activation)  97.9 -> 86.5  371 -> 356  1386 -> 1241  2406 -> 2256  8058 -> 7353
//   16384 x 2048 (activation)  38.1 -> 28.8  114 -> 97.8  435 -> 371   803 -> 663    2559 -> 2158
// Left: with all of W and A in L2 it would be 1.62 to 1.67 (its fabric's power), with
// no loads at all 2.0.  Products of 32 x 32, groups of 2 or 8 tiles along the rows
// instead of 4, starts at other stages (against channels in step), non-temporal stores
// and (with two stages) prefetches into L2 were level or slower.
#include "tile_gemm.h"

struct WideArgs {
  const bf16_t* A;                     // [M, K], row stride lda
  const bf16_t* W;                     // [N, K]
  bf16_t* C;                           // [M, N], or [M, N/2] with an activation
  int M, N, K;
  int MB, NB;                          // tiles along rows and columns
  unsigned int lda;                    // elements
};

// Which segment of 16 bytes of a row of W lies where in LDS: exclusive or with this.
// A read takes rows 8q + r (q, r < 4) of 32, so the ones that share the banks of a
// half (64 banks of 4 bytes, rows of 128 bytes) differ in bits 1, 3 and 4.
__device__ __forceinline__ int w_turn(int row) {
  return (row >> 1 & 1) | (row >> 3 & 1) << 1 | (row >> 4 & 1) << 2;
}

#define QSA_FIXED __builtin_amdgcn_sched_barrier(0)

// Tiles of 32 MT x 32 NT in blocks of 2 x 2 waves, K in stages of 64 that are loaded
// PA stages ahead: A's rows have places for so many, W's for one more.
template <int MT, int NT, int PA, int ACT>
__global__ void __launch_bounds__(256, 1) qsa_wide_gemm(WideArgs p) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int BM = 32 * MT, BN = 32 * NT;
  constexpr int TA = BM * 64, TW = BN * 64;       // elements of a stage
  constexpr int X = MT * NT / 4;                  // quartets of products, half a stage
  // a wave's loads that are younger than those of the next stage, when it waits for
  // them in the middle of one
  constexpr int AGE = (PA - 1) * NT + (PA - 2) * MT;
  constexpr int PW = PA + 1, STORES = MT * NT / (ACT ? 4 : 2);
  static_assert(NT % (ACT ? 4 : 2) == 0 && MT * NT % 4 == 0, "whole stores");
  static_assert(X >= (MT + NT) / 2 && X >= MT && X >= NT, "a slot for each load");
  __shared__ __attribute__((aligned(16))) bf16_t lds[PA * TA + PW * TW];
  bf16_t* const ldw = lds + PA * TA;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;

  // A die has a share of the tiles, of which its blocks take turns: groups of four
  // tiles along the rows, whose weights it reads together.
  const int tiles = p.MB * p.NB;
  const int die = blockIdx.x & 7, step = gridDim.x >> 3;
  int next = (int)((long long)tiles * die >> 3) + (blockIdx.x >> 3);
  const int end = (int)((long long)tiles * (die + 1) >> 3);
  if (next >= end) return;                        // uniform over the block

  // Where loads are: a tile's rows, and the stage's offset in K.  Rows and columns
  // beyond the end are zeros, and so is all beyond the last tile.
  rsrc_t ra, rw;
  int ko = 0, kstep = 0, mb = 0, nb = 0;
  auto aim = [&](int at) {
    const bool in = at < end;
    int m = 0, n = 0;
    if (in) {
      const int g = at / (4 * p.NB), r = at - g * 4 * p.NB;
      const int gm = min(4, p.MB - 4 * g);
      mb = 4 * g + r % gm;
      nb = r / gm;
      m = mb * BM;
      n = nb * (ACT ? BN / 2 : BN);
    }
    const long long ab = ((long long)(p.M - 1 - m) * p.lda + p.K) * 2;
    const long long wb = (long long)(p.N - n) * p.K * 2;
    ra = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.A + (long long)m * p.lda), 0,
        in ? (int)(unsigned)min(ab, 0xffffffffll) : 0, 0x00027000);
    rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.W + (long long)n * p.K), 0,
        in ? (int)(unsigned)min(wb, 0xffffffffll) : 0, 0x00027000);
    ko = 0;
    kstep = in ? 128 : 0;
  };
  // A load brings 8 rows of 128 bytes, a row's eight segments exchanged so that the
  // reads below spread over the banks.  Row 32 q + 8 h + 4 u + r of a wave's in LDS is
  // that column of W, with an activation column 32 (q >> 1) + 8 h + 4 (q & 1) + r of
  // the gate or (u) the up; lane (., h) of the product's tiles 2 q + u has it.
  unsigned int oa[MT], ow[NT];
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int r = (wave + j * 4) * 8 + (lane >> 3);
    oa[j] = ((unsigned)r * p.lda + ((lane & 7) ^ (r & 7)) * 8) * 2;
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int r = (wave + j * 4) * 8 + (lane >> 3);
    const int s = r % (16 * NT), q = s >> 5;      // in a wave's columns
    const unsigned int n = ACT
        ? r / (16 * NT) * (8 * NT) + (q >> 1) * 32 + (s >> 3 & 3) * 8 +
              (q & 1) * 4 + (s & 3) + (s >> 2 & 1) * (unsigned)(p.N >> 1)
        : (unsigned)r;
    ow[j] = (n * (unsigned)p.K + ((lane & 7) ^ w_turn(s)) * 8) * 2;
  }
  auto load_a = [&](int j, int place) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        ra, (lds_void_t*)(lds + place * TA + (wave + j * 4) * 512), 16, oa[j],
        ko, 0, 0);
  };
  auto load_w = [&](int j, int place) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rw, (lds_void_t*)(ldw + place * TW + (wave + j * 4) * 512), 16, ow[j],
        ko, 0, 0);
  };
  const int wm = (wave >> 1) * 16 * MT, wn = (wave & 1) * 16 * NT;
  const int wr = (col >> 2) * 8 + (col & 3);
  const bf16_t* const pa0 = lds + (wm + col) * 64;
  const bf16_t* const pw0 = ldw + (wn + wr) * 64;
  bf16x8_v fa[2][MT], fb[2][NT];
  // the x-th two of half h's operands
  auto read = [&](int h, int x, int a, int w) {
#pragma unroll
    for (int y = 2 * x; y < 2 * x + 2; ++y) {
      if (y < NT)
        fb[h][y] = *reinterpret_cast<const bf16x8_v*>(
            pw0 + ((4 * h + hi) ^ w_turn(wr)) * 8 + w * TW + (y >> 1) * 2048 +
            (y & 1) * 256);
      else if (y < NT + MT)
        fa[h][y - NT] = *reinterpret_cast<const bf16x8_v*>(
            pa0 + ((4 * h + hi) ^ (col & 7)) * 8 + a * TA + (y - NT) * 1024);
    }
  };
  f32x4_v acc[MT][NT];
  // the x-th quartet of half h: pairs of columns, down the rows and up again, each
  // product with an operand of the one before
  auto multiply = [&](int h, int x, bool first) {
#pragma unroll
    for (int z = 4 * x; z < 4 * x + 4; ++z) {
      const int b = z / (2 * MT), w = z % (2 * MT), d = w >> 1;
      const int i = b & 1 ? MT - 1 - d : d, j = 2 * b + ((w & 1) ^ (d & 1));
      acc[i][j] = mfma_bf16(fb[h][j], fa[h][i],
                            first ? (f32x4_v){0.f, 0.f, 0.f, 0.f} : acc[i][j]);
    }
  };

  int pa = 0, pw = 0;                             // places of the stage
  // Half a stage is multiplied while the next half is read.  W's loads may start with
  // the stage, in the place of the stage before; A's once all waves have read both
  // halves of this one.
  auto stage = [&](bool first, bool stores) {
    const int last = pw == 0 ? PA : pw - 1;
#pragma unroll
    for (int x = 0; x < X; ++x) {
      QSA_FIXED;
      multiply(0, x, first);
      QSA_FIXED;
      read(1, x, pa, pw);
      if ((x + 1) * NT / X > x * NT / X) load_w(x * NT / X, last);
    }
    QSA_FIXED;
    if (stores) wait_loads<(AGE + STORES > 63 ? 63 : AGE + STORES)>();
    else wait_loads<AGE>();
    stage_barrier();
    const int free = pa;
    pa = pa + 1 == PA ? 0 : pa + 1;
    pw = pw + 1 == PW ? 0 : pw + 1;
#pragma unroll
    for (int x = 0; x < X; ++x) {
      QSA_FIXED;
      multiply(1, x, false);
      QSA_FIXED;
      read(0, x, pa, pw);
      if (x < MT) load_a(x, free);
    }
    QSA_FIXED;
    ko += kstep;
  };

  aim(next);
#pragma unroll
  for (int s = 0; s < PA; ++s) {
#pragma unroll
    for (int j = 0; j < NT; ++j) load_w(j, s);
#pragma unroll
    for (int j = 0; j < MT; ++j) load_a(j, s);
    ko += kstep;
  }
  wait_loads<(PA - 1) * (MT + NT)>();
  stage_barrier();
#pragma unroll
  for (int x = 0; x < (MT + NT) / 2; ++x) read(0, x, 0, 0);
  const int steps = p.K >> 6;                     // 2 PA - 1 at least
  const int N = ACT ? p.N >> 1 : p.N;
  bool stores = false;                            // of a tile before, under way
  for (;;) {
    const int m0 = mb * BM, n0 = nb * (ACT ? BN / 2 : BN);
    stage(true, stores);
#pragma unroll
    for (int s = 1; s < PA - 1; ++s) stage(false, stores);
#pragma clang loop unroll(disable)
    for (int s = PA - 1; s < steps - PA; ++s) stage(false, false);
    next += step;
    aim(next);
#pragma unroll
    for (int s = 0; s < PA; ++s) stage(false, false);
    // a lane has columns hi * 8 .. + 7 of row `col` of each pair of tiles
    const long long left = (long long)(p.M - m0) * N * 2;
    const rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.C + (long long)m0 * N), 0,
        (int)(unsigned)min(left, 0xffffffffll), 0x00027000);
    constexpr int PS = ACT ? 4 : 2;               // tiles of a store
    const int c0 = n0 + (ACT ? wn / 2 : wn) + hi * 8;
    unsigned int to = ((unsigned)(wm + col) * N + c0) * 2;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
      for (int q = 0; q < NT / PS; ++q) {
        QSA_FIXED;
        u32x4_v v;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          f32x4_v x = acc[i][q * PS + e * PS / 2];
          if constexpr (ACT == ACT_SILU_SUM) {
            const f32x4_v u = acc[i][q * PS + e * 2 + 1];
#pragma unroll
            for (int r = 0; r < 4; ++r)
              x[r] = act_f<false, QSA_ACT_SILU>(x[r]) * u[r];
          } else if constexpr (ACT != ACT_NONE) {
            const f32x4_v u = acc[i][q * PS + e * 2 + 1];
#pragma unroll
            for (int r = 0; r < 4; ++r)
              x[r] = act_f<false, ACT - 1>(as_bf16(x[r])) * as_bf16(u[r]);
          }
          v[2 * e] = cvt_bf16x2(x[0], x[1]);
          v[2 * e + 1] = cvt_bf16x2(x[2], x[3]);
        }
        __builtin_amdgcn_raw_buffer_store_b128(
            v, rc, c0 + q * 32 < N ? to + q * 64 : 0xffffffffu, 0, 0);
      }
      to += 32u * N;
    }
    QSA_FIXED;
    if (next >= end) break;
    stores = true;
  }
  wait_loads<0>();
#endif
}

template <int MT, int NT, int PA>
static void wide_go(WideArgs p, int act, hipStream_t st) {
  p.MB = (p.M + 32 * MT - 1) / (32 * MT);
  p.NB = (p.N + 32 * NT - 1) / (32 * NT);
  const long long tiles = (long long)p.MB * p.NB;
  const dim3 grid((unsigned)(tiles < 256 ? (tiles + 7) / 8 * 8 : 256));
#define QSA_WG(ACT) \
  hipLaunchKernelGGL((qsa_wide_gemm<MT, NT, PA, ACT>), grid, dim3(256), 0, st, p)
  if constexpr (NT % 4 == 0) {
    if (act == ACT_SILU) { QSA_WG(ACT_SILU); return; }
    if (act == ACT_GELU) { QSA_WG(ACT_GELU); return; }
    if (act == ACT_SILU_SUM) { QSA_WG(ACT_SILU_SUM); return; }
  }
  QSA_WG(ACT_NONE);
#undef QSA_WG
}

// MT, NT, stages ahead; a tile's own time, a stage's where few CUs work, and one's
// where all do and the clock falls to some 1.8 GHz, us
#define QSA_WIDE(X) \
  X(8, 8, 2, 5.69f, 1.022f, 1.464f) X(6, 8, 2, 4.11f, 0.780f, 1.152f) \
  X(8, 6, 2, 4.13f, 0.781f, 1.147f) X(6, 6, 2, 3.29f, 0.622f, 0.886f) \
  X(8, 4, 3, 3.11f, 0.573f, 0.812f) X(4, 8, 2, 3.04f, 0.560f, 0.826f) \
  X(6, 4, 3, 2.48f, 0.452f, 0.647f) X(4, 6, 3, 2.59f, 0.443f, 0.643f) \
  X(4, 4, 4, 1.77f, 0.362f, 0.471f)

struct WideTile {
  int mt, nt, pa;
  float own, stage, full;
};
static const WideTile wide_tiles[] = {
#define X(MT, NT, PA, OWN, STAGE, FULL) {MT, NT, PA, OWN, STAGE, FULL},
    QSA_WIDE(X)
#undef X
};
constexpr int WIDE_TILES = sizeof(wide_tiles) / sizeof(*wide_tiles);

static float pow6(float x) { return x * x * x * x * x * x; }

// Whether a tile can do a product.
static bool wide_fits(const WideTile& t, int K, bool act) {
  return K >> 6 >= 2 * t.pa - 1 && !(act && t.nt % 4);
}

// What a tile should take for a product, us without some 2, to the power of 6: the
// turns that the blocks of a die take, the energy of all stages, or the way from memory,
// whichever binds.  Roots cost more than all the rest: only the best has one.
static float wide_pow(const WideTile& t, int M, int N, int K, bool act) {
  const int stages = K >> 6;
  const long long tiles = (long long)((M + 32 * t.mt - 1) / (32 * t.mt)) *
                          ((N + 32 * t.nt - 1) / (32 * t.nt));
  const long long turns = ((tiles + 7) / 8 + 31) / 32;
  const float own = t.own + (act ? 1.6f / 64 * (float)(t.mt * t.nt) : 0.f);
  const float run = (float)turns * (own + t.stage * (float)stages);
  const float all = t.full * (float)stages * (float)tiles * (1.f / 256);
  const float mem = 2e-6f / 5.14f * ((float)N * K + (float)M * K +
                                     (float)M * N * (act ? 0.5f : 1.f));
  return pow6(run) + pow6(all) + pow6(mem);
}
static float wide_us(float pow) { return 2.f + cbrtf(sqrtf(pow)); }

static float wide_best(int M, int N, int K, bool act, int* tile) {
  float best = INFINITY;
  for (int i = 0; i < WIDE_TILES; ++i) {
    if (!wide_fits(wide_tiles[i], K, act)) continue;
    const float pow = wide_pow(wide_tiles[i], M, N, K, act);
    if (pow < best) { best = pow; *tile = i; }
  }
  return best < INFINITY ? wide_us(best) : 1e30f;
}

// The tile that should be over first, the rows that it takes and the tile of the
// rest, if any: where the last turn would leave most blocks idle, the rows of the
// full turns are a launch of their own, which costs some 2 us beyond what the two
// should take: of 220 products the choice is then 0.5 % from the better of the two,
// 0.9 % without (us apart / in one: 18,556 x 1536 x 384 31.0 / 28.1, 5034 x 8192 x 512
// 47.7 / 44.6).  Returns us, 1e30 if K is too short for all.
extern "C" float qsa_wide_gemm_plan(int M, int N, int K, int act, int* tile,
                                    int* rows, int* rest) {
  float best = wide_best(M, N, K, act, tile);
  *rows = M;
  *rest = 0;
  for (int i = 0; i < 3; ++i) {
    const int bm = 32 * wide_tiles[i].mt, bn = 32 * wide_tiles[i].nt;
    const long long nb = (N + bn - 1) / bn, tiles = (M + bm - 1) / bm * nb;
    const int part = (int)(tiles / 256 * 256 / nb) * bm;
    if (tiles <= 256 || part == 0 || part >= M ||
        !wide_fits(wide_tiles[i], K, act))
      continue;
    const float first = wide_us(wide_pow(wide_tiles[i], part, N, K, act)) + 2.f;
    if (first >= best) continue;
    int t;
    const float us = first + wide_best(M - part, N, K, act, &t);
    if (us < best) { best = us; *tile = i; *rows = part; *rest = t; }
  }
  return best;
}

extern "C" bool qsa_wide_gemm_fits(int tile, int K, int act) {
  return tile >= 0 && tile < WIDE_TILES &&
         wide_fits(wide_tiles[tile], K, act != 0);
}

// act: 0, or an ACT_ of the first half of W's rows times the second
extern "C" void qsa_wide_gemm_launch(const bf16_t* A, const bf16_t* W, bf16_t* C,
                                     int M, int N, int K, long long lda, int tile,
                                     int act, hipStream_t st) {
  const WideArgs p{A, W, C, M, N, K, 0, 0, (unsigned int)lda};
  int i = 0;
#define X(MT, NT, PA, OWN, STAGE, FULL) \
  if (tile == i++) wide_go<MT, NT, PA>(p, act, st);
  QSA_WIDE(X)
#undef X
}
