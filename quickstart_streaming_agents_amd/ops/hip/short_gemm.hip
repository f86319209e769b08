// GEMM of a short K for CDNA4 (gfx950): C[M,N] = A[M,K] @ W[N,K]^T, bf16 with f32
// sums, and with GLU silu(gate) * up of it, W's rows being [gate; up]: the
// encoder's projections, of few rows beside rows_gemm.hip and of any where that
// module is not built.
//
// With a few steps of K a product is over before a deep pipeline is full; its
// reads and writes and, for few rows, the host's way to a library's kernel count
// as much as the matrix cores.  So: tiles by the number of blocks they leave, K in
// steps of 64 through two halves of LDS with the next one in registers, whole
// 128-byte lines of every operand, a block row's columns on one die, results
// through LDS to whole lines, and the gate's columns beside the up's in a wave, so
// that the activation costs no pass over memory.
// us, library / rows_gemm -> here:
//   384 x 512  at 100 / 400 / 1000 rows 5.4 / 5.5 / 6.2, 4.5 -> 3.1 / 3.6 / 3.8
//   1536 x 384 at 40 rows 5.0, 4.1 -> 2.8;  512 x 256 at 700 5.1, 4.0 -> 3.1
//   of few rows: qsa_few_gemm
//   at 8800 rows 1536 x 384 18.3, 17.0 -> 20.7, 384 x 512 10.7, 8.0 -> 11.7, 3072
//   x 384 with the activation 72, 30 -> 33.7
#include "lm_common.h"

struct ShortArgs {
  const bf16_t* A;                     // [M, K], row stride lda
  const bf16_t* W;                     // [N, K]
  bf16_t* C;                           // [M, N], or [M, N/2] with GLU
  int M, N, K, NB;                     // NB: blocks along the columns
  long long lda;
};

// 4 waves as 2 x 2; a wave has MT x NT tiles of 16 x 16; PF steps of K are in registers
// or under way besides the two in LDS
template <int MT, int NT, int PF, bool GLU>
__global__ void __launch_bounds__(256, 2)
qsa_short_gemm(ShortArgs p) {
  constexpr int BM = 32 * MT, BN = 32 * NT;
  constexpr int AL = BM / 32, BL = BN / 32;       // 16 B loads of a thread
  constexpr int OP = (GLU ? 8 : 16) * NT + 8;     // pitch of a wave's results
  constexpr int TILE = (BM + BN) * 64;
  __shared__ __attribute__((aligned(16))) bf16_t lds[2 * TILE];
  static_assert(4 * 16 * MT * OP <= 2 * TILE, "the results fit");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  // a die keeps the rows of a block row: it has all their columns; fewer than
  // eight block rows are spread over all dies
  const int rows = (p.M + BM - 1) / BM;
  int mb, nb;
  if (rows < 8) {
    mb = blockIdx.x % rows;
    nb = blockIdx.x / rows;
  } else {
    mb = (blockIdx.x / 8 / p.NB) * 8 + blockIdx.x % 8;
    nb = blockIdx.x / 8 % p.NB;
    if (mb >= rows) return;            // uniform over the block
  }
  const int m0 = mb * BM;

  // thread: 16 bytes of row tid/8 (+ 32 j), the eight of a row side by side
  const int seg = tid & 7, r8 = tid >> 3;
  const bf16_t* ap[AL];
  const bf16_t* bp[BL];
#pragma unroll
  for (int j = 0; j < AL; ++j)
    ap[j] = p.A + (long long)min(m0 + r8 + 32 * j, p.M - 1) * p.lda + seg * 8;
#pragma unroll
  for (int j = 0; j < BL; ++j) {
    const int r = r8 + 32 * j;         // row of the tile
    int n = nb * BN + r;
    if (GLU)                           // tiles 2i and 2i + 1: gate, up
      n = (r >> 4 & 1) * (p.N >> 1) + nb * (BN / 2) + (r >> 5) * 16 + (r & 15);
    bp[j] = p.W + (long long)min(n, p.N - 1) * p.K + seg * 8;
  }
  // LDS: fragments [row tile][half of K][hi][16 rows][8], the rows of a group
  // exchanged so that a row's eight segments go to different banks
  auto place = [&](int row, int half, int h) {
    return (((row >> 4) * 2 + half) * 64 + h * 16 +
            ((row & 15) ^ (h << 1 | half << 3))) * 8;
  };
  u32x4_v ar[PF][AL], br[PF][BL];
  const int steps = p.K >> 6;
  auto load = [&](int q, int step) {   // beyond the end: the last one again
    const int k = min(step, steps - 1) * 64;
#pragma unroll
    for (int j = 0; j < AL; ++j)
      ar[q][j] = *reinterpret_cast<const u32x4_v*>(ap[j] + k);
#pragma unroll
    for (int j = 0; j < BL; ++j)
      br[q][j] = *reinterpret_cast<const u32x4_v*>(bp[j] + k);
  };
  auto store = [&](int q, bf16_t* t) {
#pragma unroll
    for (int j = 0; j < AL; ++j)
      *reinterpret_cast<u32x4_v*>(
          t + place(r8 + 32 * j, seg >> 2, seg & 3)) = ar[q][j];
#pragma unroll
    for (int j = 0; j < BL; ++j)
      *reinterpret_cast<u32x4_v*>(
          t + BM * 64 + place(r8 + 32 * j, seg >> 2, seg & 3)) = br[q][j];
  };
  f32x4_v acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  const int wm = (wave >> 1) * MT, wn = (wave & 1) * NT;
  auto step = [&](int s, int q) {      // q: where the next step's registers are
    lds_barrier();
    const bf16_t* t = lds + (s & 1) * TILE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8_v a[MT], b[NT];
      const int at = h * 512 + (hi * 16 + (col ^ (hi << 1 | h << 3))) * 8;
#pragma unroll
      for (int i = 0; i < MT; ++i)
        a[i] = *reinterpret_cast<const bf16x8_v*>(t + (wm + i) * 1024 + at);
#pragma unroll
      for (int j = 0; j < NT; ++j)
        b[j] = *reinterpret_cast<const bf16x8_v*>(t + BM * 64 +
                                                  (wn + j) * 1024 + at);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = mfma_bf16(b[j], a[i], acc[i][j]);
    }
    if (PF > 1 || s + 1 < steps) {     // no branch around loads that are counted
      store(q, lds + ((s + 1) & 1) * TILE);       // behind the last: not read
      load(q, s + 1 + PF);
    }
  };
#pragma unroll
  for (int q = 0; q < PF; ++q) load(q, q);
  store(0, lds);
  load(0, PF);
  int s = 0;
  for (; s + PF <= steps; s += PF)
#pragma unroll
    for (int q = 0; q < PF; ++q) step(s + q, (q + 1) % PF);
#pragma unroll
  for (int q = 0; q < PF - 1; ++q)
    if (s + q < steps) step(s + q, (q + 1) % PF); // uniform over the block
  // results through LDS: a lane has 4 columns (hi*4..) of row col of each tile
  lds_barrier();
  bf16_t* o = lds + wave * (16 * MT * OP);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; j += GLU ? 2 : 1) {
      f32x4_v v = acc[i][j];
      if constexpr (GLU) {
        const f32x4_v u = acc[i][j + 1];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = v[r] / (1.f + __expf(-v[r])) * u[r];
      }
      *reinterpret_cast<uint2*>(
          o + (i * 16 + col) * OP + (GLU ? j / 2 : j) * 16 + hi * 4) =
          make_uint2(cvt_bf16x2(v[0], v[1]), cvt_bf16x2(v[2], v[3]));
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  constexpr int G = (GLU ? NT : 2 * NT);          // 16 B groups of a row
  const int N = GLU ? p.N >> 1 : p.N;
  const int c0 = (GLU ? nb * (BN / 2) : nb * BN) + (wave & 1) * G * 8;
#pragma unroll
  for (int i = lane; i < 16 * MT * G; i += 64) {
    const int row = i / G, c = (i % G) * 8;
    const int m = m0 + (wave >> 1) * 16 * MT + row;
    if (m < p.M && c0 + c < N)                    // N % 8 == 0
      *reinterpret_cast<u32x4_v*>(p.C + (long long)m * N + c0 + c) =
          *reinterpret_cast<const u32x4_v*>(o + row * OP + c);
  }
}

// Few rows: 8 waves of a block share K, for 32 rows x 16 columns (with GLU of gate and
// up each), and all of a wave's operands are on their way to registers at once, so that
// a product is one latency of memory and a sum in LDS, where the tiles above wait for a
// barrier every 64 of K.
template <int U, bool GLU>
__global__ void __launch_bounds__(512)
qsa_few_gemm(ShortArgs p) {
  constexpr int NW = 8, T = GLU ? 2 : 1, PITCH = 68;     // banks of a row's sums differ
  __shared__ float red[NW][T * 8 * PITCH];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 32;
  const int steps = p.K >> 6;
  const bf16_t *ap[2], *bp[T];
#pragma unroll
  for (int m = 0; m < 2; ++m)
    ap[m] = p.A + (long long)min(m0 + m * 16 + col, p.M - 1) * p.lda + hi * 8;
#pragma unroll
  for (int t = 0; t < T; ++t)
    bp[t] = p.W + (long long)(n0 + col + t * (p.N >> 1)) * p.K + hi * 8;
  f32x4_v acc[T][2];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int m = 0; m < 2; ++m) acc[t][m] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  for (int s = wave; s < steps; s += NW * U) {
    bf16x8_v a[U][2][2], b[U][T][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(s + u * NW, steps - 1) * 64;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int t = 0; t < T; ++t)
          b[u][t][i] = *reinterpret_cast<const bf16x8_v*>(bp[t] + k + i * 32);
#pragma unroll
        for (int m = 0; m < 2; ++m)
          a[u][m][i] = *reinterpret_cast<const bf16x8_v*>(ap[m] + k + i * 32);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u * NW >= steps) break;             // uniform over the wave
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
          for (int m = 0; m < 2; ++m)
            acc[t][m] = mfma_bf16(b[u][t][i], a[u][m][i], acc[t][m]);
    }
  }
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wave][((t * 2 + m) * 4 + r) * PITCH + lane] = acc[t][m][r];
  __syncthreads();
  // a lane had columns hi * 4 .. + 3 of row `col`; a thread takes one number
  const int row = tid >> 4, c = tid & 15;
  const int at = ((row >> 4) * 4 + (c & 3)) * PITCH + (c >> 2) * 16 + (row & 15);
  float v[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    v[t] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v[t] += red[w][t * 8 * PITCH + at];
  }
  if constexpr (GLU) v[0] = v[0] / (1.f + __expf(-v[0])) * v[T - 1];
  if (m0 + row < p.M)
    p.C[(long long)(m0 + row) * (GLU ? p.N >> 1 : p.N) + n0 + c] = cvt_bf16(v[0]);
}

template <int U>
static void few_go(const ShortArgs& p, int glu, hipStream_t st) {
  const dim3 grid((unsigned)(p.N / (glu ? 32 : 16)), (unsigned)((p.M + 31) / 32));
  if (glu)
    hipLaunchKernelGGL((qsa_few_gemm<U, true>), grid, dim3(512), 0, st, p);
  else
    hipLaunchKernelGGL((qsa_few_gemm<U, false>), grid, dim3(512), 0, st, p);
}

template <int MT, int NT, int PF = 1>
static void short_go(ShortArgs p, int glu, hipStream_t st) {
  p.NB = (p.N + 32 * NT - 1) / (32 * NT);
  const int mb = (p.M + 32 * MT - 1) / (32 * MT);
  const dim3 grid((unsigned)((mb < 8 ? mb : (mb + 7) / 8 * 8) * p.NB));
  if (glu)
    hipLaunchKernelGGL((qsa_short_gemm<MT, NT, PF, true>), grid, dim3(256), 0, st,
                       p);
  else
    hipLaunchKernelGGL((qsa_short_gemm<MT, NT, PF, false>), grid, dim3(256), 0, st,
                       p);
}

// Blocks of 32 rows and 16 columns while each has a CU to itself, with the gate's half
// of them (us, tiles / so: 1536 x 384 of 15 rows 3.21 / 2.59, of 60, 192 blocks, 3.24 /
// 2.92, of 130, 480 blocks, 3.30 / 4.06; 384 x 1536 of 15 rows 7.2 / 4.7, of 250, 192
// blocks, 7.4 / 5.9, of 400, 312 blocks, 7.4 / 9.8; gated 1536 x 384 of 15 rows 3.31 /
// 3.00, of 60, 96 blocks, 3.34 / 3.36, of 130, 240 blocks, 3.37 / 3.46).
static bool few_takes(long long M, long long N, bool glu) {
  return (M + 31) / 32 * (N / (glu ? 32 : 16)) <= (glu ? 128 : 256);
}

// Which of the encoder's products are this file's where rows_gemm.hip and wide_gemm.hip
// are there too: while the tiles of 32 x 64 leave CUs idle, K being short or the rows
// few (the figures above and at the encoder's products).
extern "C" bool qsa_short_gemm_takes(long long M, long long N, long long K) {
  return K % 64 == 0 && N % 32 == 0 && N < 1 << 20 && (K <= 512 || M <= 32) &&
         (M + 31) / 32 * ((N + 63) / 64) <= 192;
}

// Tiles of 128 x 128 once two rounds of blocks are left, 64 x 64 while they
// make half a round, 32 x 64 below (384 x 512 at 400 rows: 8.2 / 4.5 / 3.7 us;
// 1536 x 384 at 1600: 7.9 / 6.8 / 8.0, at 8800: 20.9 / 23.0 / 28.4; 3072 x 384
// with the activation at 16,000: 58 with 128 x 128, 94 with 32 x 64).  Six steps of K
// ahead pay where K is long (384 x 1536 of 15 rows 7.2 -> 6.2 us); a few are over by
// then, and as many more are read in vain (one ahead / six: 1536 x 384 at 130 and 320
// rows 3.57 / 3.69, 4.41 / 5.02, 3072 x 384 gated at 100 3.76 / 3.94, 384 x 128 at 600
// 2.76 / 3.10; K 512 level).
extern "C" void qsa_short_gemm_launch(const bf16_t* A, const bf16_t* W,
                                      bf16_t* C, int M, int N, int K,
                                      long long lda, int glu,
                                      hipStream_t st) {
  if (M == 0) return;
  const ShortArgs p{A, W, C, M, N, K, 0, lda};
  auto blocks = [&](int b) {
    return (long long)((M + b - 1) / b) * ((N + b - 1) / b);
  };
  if (few_takes(M, N, glu)) {
    if (K <= 512) few_go<1>(p, glu, st); else few_go<3>(p, glu, st);
    return;
  }
  if (blocks(128) >= 512) short_go<4, 4>(p, glu, st);
  else if (blocks(64) >= 128) short_go<2, 2>(p, glu, st);
  else if (K <= 512) short_go<1, 2>(p, glu, st);
  else short_go<1, 2, 6>(p, glu, st);
}
