// GEMM on weights as they are stored, for decode batches, short prompts and all
// else that leaves a library's large tiles idle: C[M,N] = A[M,K] @ W[N,K]^T, bf16
// with f32 sums, or act(gate) * up of it with W = [gate; up].
//
// Up to some 200 rows it is bound by the read of W, then by the matrix cores.
// Both operands go from memory straight into LDS (16 bytes a lane, whole lines),
// through a ring of two to six stages of K, as deep as the 160 KB of a CU allow, so
// the bytes under way do not cost registers.  A wave multiplies half a
// stage while it reads the next half.  Tiles from 64 x 32 to 256 x 256 and
// shares of K are chosen by what they should take (qsa_rows_gemm_plan); a tile's
// LDS traffic per product falls with its sides, which is why the large ones are
// the fast ones where the chip is full.  The activation
// is applied to the sums, rounded first where a stored product was read before.
// us, library -> here (sums of shares included, weights from memory):
//   rows            33            64           128           192           768
//   6144 x 4096  17.2 -> 15.7  18.0 -> 17.3  25.7 -> 22.6  33.5 -> 27.3  48 -> 46
//   4096 x 4096  13.9 -> 11.4  15.4 -> 12.9  24.8 -> 16.5  32.9 -> 19.3  34 -> 35
//   4096 x 14336 34.6 -> 26.4  39.2 -> 27.5  75.7 -> 36.4   103 -> 45   107 -> 95
//   2048 x 8192  14.1 -> 12.3  22.6 -> 13.4  21.1 -> 16.0  26.5 -> 19.7  43 -> 36
//   12576 x 2048 16.6 -> 12.9  16.5 -> 14.3  19.3 -> 18.3  26.0 -> 22.4  42 -> 47
// with the activation (there a pass of its own):
//   28672 x 4096 53.3 -> 43.0  53.5 -> 43.0  57.1 -> 51.2  66.4 -> 59.3 167 -> 180
//   16384 x 2048 21.9 -> 14.3  20.9 -> 15.3  24.0 -> 19.2  30.6 -> 23.6  53 -> 52
// What limits 256 x 256 at 1.3 PFLOP/s is the loads' latency with two stages in LDS;
// products that fill the chip are wide_gemm.hip's.
#include "tile_gemm.h"

struct RowsArgs {
  const bf16_t* A;                     // [M, K], row stride lda
  const bf16_t* W;                     // [N, K]
  bf16_t* C;                           // [M, N], or [M, N/2] with an activation
  float* part;                         // [S][M][N] where S > 1
  int M, N, K, S;
  int MB, NB;                          // blocks along rows and columns
  unsigned int lda;                    // elements
  bool far;                            // W is larger than the last-level cache,
                                       // together with what a step reads beside it
};

// Whether two blocks of eight waves share a CU's 160 KB (128 bytes a row and stage)
constexpr bool rows_pair(int bm, int bn, int waves, int st) {
  return waves == 8 && st * (bm + bn) * 128 <= 80 * 1024;
}

// BM x BN of C in a block of WM x WN waves, K in stages of 64 through a ring of
// ST places in LDS; with ACT, W's rows are [gate; up] and a wave's column tiles
// are alternately of either.
// ONCE: W's loads leave no trace in the last-level cache (see the launch).
template <int BM, int BN, int WM, int WN, int ST, int ACT, bool ONCE>
__global__ void __launch_bounds__(WM * WN * 64,
                                  rows_pair(BM, BN, WM * WN, ST) ? 4 : 1)
qsa_rows_gemm(RowsArgs p) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int NW = WM * WN, MT = BM / WM / 16, NT = BN / WN / 16;
  constexpr int STAGE = (BM + BN) * 64;           // elements
  constexpr int L = (BM + BN) / 8 / NW;           // loads of a wave and stage
  constexpr int AL = BM / 8 / NW;                 // of them A's
  constexpr int RD = MT + NT, MM = MT * NT;       // reads, MFMAs of half a stage
  constexpr int OP = (ACT ? 8 : 16) * NT + 8;     // pitch of a wave's results
  constexpr int OUT = NW * MT * 16 * OP;
  static_assert(BM / 8 % NW == 0 && BN / 8 % NW == 0, "whole loads");
  static_assert(!ACT || NT % 2 == 0, "pairs of column tiles");
  __shared__ __attribute__((aligned(16)))
      bf16_t lds[ST * STAGE > OUT ? ST * STAGE : OUT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;

  // A die takes neighbouring work: one share of K, then groups of four block
  // rows, whose weights it reads together.
  const int per = gridDim.x >> 3, tiles = p.MB * p.NB;
  const int at = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (at >= tiles * p.S) return;                  // uniform over the block
  const int share = at / tiles, t = at - share * tiles;
  const int g = t / (4 * p.NB), gm = min(4, p.MB - 4 * g);
  const int mb = 4 * g + (t - 4 * g * p.NB) % gm;
  const int nb = (t - 4 * g * p.NB) / gm;
  const int m0 = mb * BM, n0 = nb * BN;
  const int all = p.K >> 6;
  const int s0 = (int)((long long)all * share / p.S);
  const int steps = (int)((long long)all * (share + 1) / p.S) - s0;
  // Where a block starts in its share: rows of W lie a multiple of the memory
  // channels' period apart, so blocks in step would meet in the same channels
  // (28672 x 4096 at 64 rows: 56 us in step, 46 in turn).  Many block rows share
  // the columns through L2 instead.
  const int turn = p.MB > 2 ? 0 : (int)((long long)nb * steps / p.NB);

  const rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.A + (long long)m0 * p.lda + s0 * 64), 0, 0xffffffffu,
      0x00027000);
  const rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.W + (long long)(ACT ? n0 / 2 : n0) * p.K + s0 * 64), 0,
      0xffffffffu, 0x00027000);
  // A load brings 8 rows of 128 bytes, a row's eight segments exchanged by its
  // number so that the reads below spread over the banks.  Rows and columns
  // beyond the end shadow the last one and are not stored.
  unsigned int off[L];
#pragma unroll
  for (int j = 0; j < L; ++j) {
    const int r = (wave + j * NW) * 8 + (lane >> 3);
    const int seg = (lane & 7) ^ (r & 7);
    if (j < AL) {
      off[j] = ((unsigned)min(r, p.M - 1 - m0) * p.lda + seg * 8) * 2;
    } else {
      const int q = r - BM;
      const int n = ACT ? min((q >> 5) * 16 + (q & 15),
                              (p.N - n0) / 2 - 1) + (q >> 4 & 1) * (p.N >> 1)
                        : min(q, p.N - 1 - n0);
      off[j] = ((unsigned)n * (unsigned)p.K + seg * 8) * 2;
    }
  }
  auto load = [&](int s, int place) {
    const int k = s + turn < steps ? s + turn : s + turn - steps;
#pragma unroll
    for (int j = 0; j < L; ++j)
      if (j < AL)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            ra, (lds_void_t*)(lds + place * STAGE + (wave + j * NW) * 512), 16,
            off[j], k * 128, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rw, (lds_void_t*)(lds + place * STAGE + (wave + j * NW) * 512), 16,
            off[j], k * 128, 0, ONCE ? QSA_NT : 0);
  };
  const int wm = wave / WN * MT, wn = wave % WN * NT;
  bf16x8_v fa[2][MT], fb[2][NT];
  auto read = [&](int h, int place) {
    const bf16_t* b = lds + place * STAGE + col * 64 +
                      ((h * 4 + hi) ^ (col & 7)) * 8;
#pragma unroll
    for (int j = 0; j < NT; ++j)
      fb[h][j] = *reinterpret_cast<const bf16x8_v*>(b + BM * 64 +
                                                    (wn + j) * 1024);
#pragma unroll
    for (int i = 0; i < MT; ++i)
      fa[h][i] = *reinterpret_cast<const bf16x8_v*>(b + (wm + i) * 1024);
  };
  f32x4_v acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int h) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = mfma_bf16(fb[h][j], fa[h][i], acc[i][j]);
  };

  // Half a stage is multiplied while the next half is read.  Once both of a
  // stage are in registers its place takes the stage ST further on.
#pragma unroll
  for (int s = 0; s < ST; ++s)
    if (s < steps) load(s, s);
  if (steps >= ST) wait_loads<(ST - 1) * L>();
  else wait_loads<0>();
  stage_barrier();
  read(0, 0);
  int place = 0, s = 0;
  for (; s < steps - ST; ++s) {
    read(1, place);
    multiply(0);
#pragma unroll
    for (int i = 0; i < RD; ++i) {     // a read every few MFMAs
      __builtin_amdgcn_sched_group_barrier(0x8, MM / RD ? MM / RD : 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    wait_loads<(ST - 2) * L>();        // stage s + 1 is there
    stage_barrier();
    load(s + ST, place);
    place = place + 1 == ST ? 0 : place + 1;
    read(0, place);
    multiply(1);
    constexpr int PM = MM / (RD + L) ? MM / (RD + L) : 1;
#pragma unroll
    for (int i = 0; i < (RD > L ? RD : L); ++i) {
      if (i < L) {
        __builtin_amdgcn_sched_group_barrier(0x8, PM, 0);
        __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
      }
      if (i < RD) {
        __builtin_amdgcn_sched_group_barrier(0x8, PM, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  for (; s < steps; ++s) {             // no more loads: those under way
    read(1, place);
    multiply(0);
    const int ahead = steps - 2 - s;   // stages that may still be under way
    if (ahead >= ST - 2) wait_loads<(ST - 2) * L>();
    else if (ST > 3 && ahead == ST - 3) wait_loads<(ST > 3 ? ST - 3 : 0) * L>();
    else if (ST > 4 && ahead == ST - 4) wait_loads<(ST > 4 ? ST - 4 : 0) * L>();
    else if (ST > 5 && ahead == ST - 5) wait_loads<(ST > 5 ? ST - 5 : 0) * L>();
    else wait_loads<0>();
    stage_barrier();
    place = place + 1 == ST ? 0 : place + 1;
    read(0, place);                    // after the last stage: not used
    multiply(1);
  }

  // a lane has columns hi * 4 .. + 3 of row `col` of each tile
  if (p.S > 1) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = m0 + (wm + i) * 16 + col;
      if (row >= p.M) continue;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int c = n0 + (wn + j) * 16 + hi * 4;          // N % 16 == 0
        if (c < p.N)
          *reinterpret_cast<f32x4_v*>(
              p.part + ((long long)share * p.M + row) * p.N + c) = acc[i][j];
      }
    }
    return;
  }
  // results through LDS to whole lines; the last reads above are in a wave's
  // own registers, so its barrier suffices
  wait_loads<0>();
  stage_barrier();
  bf16_t* o = lds + wave * (MT * 16 * OP);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; j += ACT ? 2 : 1) {
      f32x4_v v = acc[i][j];
      if constexpr (ACT == ACT_SILU_SUM) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = act_f<false, QSA_ACT_SILU>(v[r]) * acc[i][j + 1][r];
      } else if constexpr (ACT != ACT_NONE) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = act_f<false, ACT - 1>(as_bf16(v[r])) *
                 as_bf16(acc[i][j + 1][r]);
      }
      *reinterpret_cast<uint2*>(o + (i * 16 + col) * OP +
                                (ACT ? j / 2 : j) * 16 + hi * 4) =
          make_uint2(cvt_bf16x2(v[0], v[1]), cvt_bf16x2(v[2], v[3]));
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  constexpr int G = ACT ? NT : 2 * NT;            // 16 B groups of a row
  const int N = ACT ? p.N >> 1 : p.N;
  const int c0 = (ACT ? n0 / 2 : n0) + wave % WN * G * 8;
#pragma unroll
  for (int x = 0; x < (MT * G + 3) / 4; ++x) {
    const int i = x * 64 + lane, row = i / G, c = i % G * 8;
    const int m = m0 + wm * 16 + row;
    if (row < MT * 16 && m < p.M && c0 + c < N)   // N % 8 == 0
      *reinterpret_cast<u32x4_v*>(p.C + (long long)m * N + c0 + c) =
          *reinterpret_cast<const u32x4_v*>(o + row * OP + c);
  }
#endif
}

__global__ void __launch_bounds__(256)
qsa_rows_sum(const float* __restrict__ part, bf16_t* __restrict__ C,
             long long n, int S) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;                  // n % 4 == 0
  float v[4];
  ld_shares<4>(part + i, n, S, v);
  *reinterpret_cast<uint2*>(C + i) =
      make_uint2(cvt_bf16x2(v[0], v[1]), cvt_bf16x2(v[2], v[3]));
}

template <int BM, int BN, int WM, int WN, int ST>
static void rows_go(RowsArgs p, int act, hipStream_t st) {
  p.MB = (p.M + BM - 1) / BM;
  p.NB = (p.N + BN - 1) / BN;
  const dim3 grid((unsigned)((long long)p.MB * p.NB * p.S + 7) / 8 * 8);
  // One block row reads every weight once, and the weights of a step's other layers
  // drive it out of the last-level cache before the next step; past it they come faster
  // and leave it to what fits (decoder of width 4096, 8 layers, 192 rows of 400-1000
  // keys 2295 -> 2180 us a step with keys and values likewise, 28672 x 4096 57 -> 54;
  // of width 2048, 64 rows 813 -> 746).
  const bool once =
      p.far && BM <= 192 && p.MB == 1 && (long long)p.N * p.K >= 2 << 20;
#define QSA_RG_AS(ACT, ONCE) \
  hipLaunchKernelGGL((qsa_rows_gemm<BM, BN, WM, WN, ST, ACT, ONCE>), grid, \
                     dim3(WM * WN * 64), 0, st, p)
#define QSA_RG(ACT) \
  if constexpr (BM <= 192) { \
    if (once) QSA_RG_AS(ACT, true); else QSA_RG_AS(ACT, false); \
  } else { \
    QSA_RG_AS(ACT, false); \
  }
  if constexpr (BN / WN / 16 % 2 == 0) {
    if (act == ACT_SILU) { QSA_RG(ACT_SILU) return; }
    if (act == ACT_GELU) { QSA_RG(ACT_GELU) return; }
    if (act == ACT_SILU_SUM) { QSA_RG(ACT_SILU_SUM) return; }
  }
  QSA_RG(ACT_NONE)
#undef QSA_RG_AS
#undef QSA_RG
}

// BM, BN, waves, places of the ring; a block's own time and that of a stage, us, and
// the same where few rows meet weights from memory (qsa_rows_gemm_plan).
// Of the last tile two blocks share a CU: one's start and end lie beside the
// other's products, which short K gains by (us, the best of the others and so:
// 16,000 x 3072 x 384 with the activation 52.7, 49.3; 24,000 79.2, 71.7; 8263 x
// 2048 x 128 15.7, 13.0; 30,000 38.2, 30.7; 4400 x 16384 x 2048 263, 253).  Its
// figures are those of a pair, set where 42 such shapes part.
#define QSA_TILES(X) \
  X(64, 32, 2, 2, 6, 0.67f, 0.200f, 1.04f, 0.178f) \
  X(64, 64, 2, 2, 4, 0.71f, 0.208f, 1.40f, 0.235f) \
  X(64, 128, 2, 4, 6, 1.86f, 0.353f, 3.17f, 0.377f) \
  X(128, 64, 4, 2, 6, 1.92f, 0.334f, 3.39f, 0.309f) \
  X(128, 128, 2, 4, 4, 2.38f, 0.497f, 4.44f, 0.438f) \
  X(192, 64, 4, 2, 4, 1.94f, 0.431f, 3.05f, 0.456f) \
  X(192, 128, 4, 2, 4, 2.98f, 0.644f, 5.12f, 0.592f) \
  X(256, 128, 4, 2, 3, 3.41f, 0.822f, 4.68f, 0.688f) \
  X(128, 256, 2, 4, 3, 3.32f, 0.843f, 6.16f, 0.712f) \
  X(192, 192, 2, 4, 3, 4.03f, 0.800f, 6.82f, 0.674f) \
  X(256, 192, 4, 2, 2, 3.57f, 1.189f, 3.45f, 1.160f) \
  X(192, 256, 2, 4, 2, 3.19f, 1.227f, 5.16f, 1.223f) \
  X(256, 256, 2, 4, 2, 4.06f, 1.482f, 3.51f, 1.350f) \
  X(192, 128, 4, 2, 2, 0.77f, 1.27f, 2.31f, 0.956f)

struct RowsTile {
  int bm, bn, wn;
  bool pair;                           // of large blocks on a CU
  float own, stage, own_few, stage_few;
};
static const RowsTile rows_tiles[] = {
#define X(BM, BN, WM, WN, ST, OWN, STAGE, OWN2, STAGE2)                \
  {BM, BN, WN, rows_pair(BM, BN, WM * WN, ST), OWN, STAGE, OWN2, STAGE2},
    QSA_TILES(X)
#undef X
};

// The tile and the shares of K that should be over first.  Blocks take turns on
// the 256 CUs, a turn as long as its stages or the whole product's way from
// memory, whichever binds; shares cost the writing and adding of their sums.
// The figures above and here are fitted to 382 shapes at up to 20 tiles and
// shares each (M 33 to 20000, N 128 to 32000, K 128 to 14336; off by 9 % each,
// and the choice by 1 % from the best of them).  Two blocks of the smallest
// tiles share a CU, so a stage takes another time alone on it.  The one of 64 x 32,
// which fetches two rows of A with every row of W, follows 368 more shapes (M 1 to
// 20,000, N 96 to 57,000): at 0.141 a stage beside another block it was the choice
// for 64 x 12288 x 8192 (60 us for 45, the library 46) and 64 x 16384 x 2048 (21
// for 15).  Over these the choice is 2.5 % from the best, 5.1 before, and 18 of
// them, 37 before, are more than 5 % behind the library, the larger by up to 14 %
// (450 to 512 x 12288, 64 x 40960 x 12288).
// Few rows are another matter: their weights come from memory, each block's rows of A
// once more from L2, and what a CU gets through it binds (192 x 6144 x 4096, us: 192 x
// 64 in two shares 28.2, for which the figures above say 22.7, 128 x 64 whole 24.2;
// 192 x 4096 x 14336: 192 x 64 in four 42.9, 192 x 128 in eight 37.0).  For 81 to
// 192 rows and from 2M weights on the tiles' second figures are fitted to 1722 times of
// 84 shapes (weights in turn from 700 MB): off by 6 %, and the choice 1.0 % from the
// best, 3.3 % with the figures above; a decoder's step of
// width 4096, 8 layers, 192 rows 2166 -> 2081 us, of 150 1644 -> 1614, of 100 1354 -> 1339,
// but of 66 1146 -> 1152.
// cheap: the reader of the product adds the shares; us_out: what the choice should
// take, or null.
extern "C" int qsa_rows_gemm_plan(int M, int N, int K, int act, int cheap,
                                  int* shares, float* us_out) {
  const int all = K >> 6;
  const bool few = M > 80 && M <= 192 && (long long)N * K >= 2 << 20;
  const float mem = 2e-6f / (few ? 7.06f : 5.14f) *
                    ((float)N * K + (float)M * K + (float)M * N);
  const float sum = few ? (cheap ? 1.22f : 3.79f) : (cheap ? 0.5f : 3.25f);
  const float each = (few ? 1.40e-6f : 1.28e-6f) * (float)M * N;
  float best = 1e30f;
  int tile = 0;
  *shares = 1;
  for (int i = 0; i < (int)(sizeof(rows_tiles) / sizeof(*rows_tiles)); ++i) {
    const RowsTile& t = rows_tiles[i];
    if (act && t.bn / t.wn / 16 % 2) continue;    // no pairs of column tiles
    const long long blocks =
        (long long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    if (t.pair && blocks <= 256) continue;        // alone on their CUs
    const int fill = blocks < 256 ? (int)(256 / blocks) : 1;
    int most = act || all < 8 ? 1 : fill;
    if (few)                           // 1, 2, 4 or 8
      for (most = std::min(most, 8); most & (most - 1); --most) {}
    for (int S = most; S >= 1; S = S > 1 ? S / 2 : 0) {
      if (S > all / 4 && S > 1) continue;
      const int slots = t.pair ? 512 : 256;
      const long long turns = (blocks * S + slots - 1) / slots;
      float stage = few ? t.stage_few : t.stage;
      if (turns == 1 && t.bn * t.bm <= 4096)
        stage *= few ? (i ? 1.26f : 1.39f) : (i ? 1.48f : 0.93f);
      float run = (float)turns * ((few ? t.own_few : t.own) +
                                  stage * ((all + S - 1) / S));
      if (t.pair && turns == 1) run += 1.5f;      // neither end beside another
      const float after = S > 1 ? sum + each * S : 0.f;
      if (run + after >= best) continue;          // no root makes it less
      const float r2 = run * run, m2 = mem * mem;
      const float us =
          (few ? sqrtf(r2 + m2) : sqrtf(sqrtf(r2 * r2 + m2 * m2))) + after;
      if (us < best) { best = us; tile = i; *shares = S; }
    }
  }
  if (us_out) *us_out = best;
  return tile;
}

// act: 0, or an ACT_ of the first half of W's rows times the second (one share
// only).  With part and S > 1 and no C the shares are left to the caller.
extern "C" void qsa_rows_gemm_launch(const bf16_t* A, const bf16_t* W,
                                     bf16_t* C, float* part, int M, int N,
                                     int K, long long lda, int tile, int S,
                                     int act, bool far, hipStream_t st) {
  const RowsArgs p{A, W, C, part, M, N, K, S, 0, 0, (unsigned int)lda, far};
  int i = 0;
#define X(BM, BN, WM, WN, ST, OWN, STAGE, OWN2, STAGE2) \
  if (tile == i++) rows_go<BM, BN, WM, WN, ST>(p, act, st);
  QSA_TILES(X)
#undef X
  if (S > 1 && C) {
    const long long n = (long long)M * N;
    hipLaunchKernelGGL(qsa_rows_sum, dim3((unsigned)((n / 4 + 255) / 256)),
                       dim3(256), 0, st, part, C, n, S);
  }
}
