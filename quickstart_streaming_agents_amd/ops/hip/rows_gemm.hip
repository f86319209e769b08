// Decode-batch GEMM on weights as they are stored, for a projection from many
// columns to few: C[M,N] = A[M,K] @ W[N,K]^T, 32 < M <= 192 rows, K >= 3 N,
// bf16 with f32 sums.
//
// Bound by the read of W; what stands in the way is that N alone makes too few
// blocks, and that the rows, read again by every block, cost as much cache
// bandwidth as W once there are many of them.  So K is split until every CU has
// a block, each block keeps all rows of its share (A passes through LDS once
// for its four waves), and W goes from memory to the matrix cores' operands
// directly, 32 columns a wave, 128 bytes of each at a time.  The shares' sums
// meet in f32 in a second kernel.
// us, library GEMM -> here (sums included, weights from memory), at 40 / 64 /
// 128 / 192 rows:
//   2048 x  8192  14.1 / 22.6 / 21.1 / 26.5 -> 14.7 / 15.4 / 21.0 / 25.9
//   2560 x  8192  16.3 / 23.1 / 41.8 / 26.9 -> 17.5 / 18.7 / 25.1 / 30.9
//   1536 x 11264  20.8 / 31.0 / 27.2 / 38.2 -> 16.9 / 18.1 / 24.1 / 30.1
//   2560 x 10240  20.9 / 30.5 / 55.8 / 36.7 -> 19.5 / 21.2 / 27.8 / 34.7
//   4096 x 14336  36.7 / 41.2 / 76.2 / 64.3 -> 29.1 / 32.0 / 42.1 / 54.6
//   4096 x 16384  38.8 / 42.5 / 82.4 / 115  -> 39.5 / 39.8 / 48.3 / 58.3
//   5120 x 15360  49.7 / 53.9 / 82.8 / 112  -> 40.0 / 43.4 / 54.8 / 68.4
//   8192 x 24576   113 /  130 /  181 /  210 ->  104 /  113 /  130 /  159
// With N nearer to K the library's larger tiles win: 4096 x 4096 at 192 rows
// 20.5 against 25.6, 16384 x 2048 27.2 against 36.
#include "lm_common.h"

struct RowsArgs {
  const bf16_t* A;
  const bf16_t* W;
  float* part;                         // [S][M][N]
  int M, N, K;
  unsigned int lda;                    // elements
};

// 64 of K a step; two steps of A and W are under way in registers
template <int MT>                      // row tiles of 16
__global__ void __launch_bounds__(256)
qsa_rows_gemm(RowsArgs p) {
  constexpr int CT = 2, D = 2;         // column tiles of a wave, steps ahead
  constexpr int AF = MT * 2;           // fragments of A a step
  constexpr int AL = (AF + 3) / 4;     // and of them per wave
  __shared__ __attribute__((aligned(16))) bf16_t at[2][AF * 512];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  const int n0 = (blockIdx.x * 4 + wave) * 16 * CT;
  const int steps = p.K >> 6, S = gridDim.y;      // K % 64 == 0, S <= steps
  const int s0 = (int)((long long)steps * blockIdx.y / S);
  const int s1 = (int)((long long)steps * (blockIdx.y + 1) / S);

  // rows and columns beyond the end shadow the last one and are not stored
  unsigned int aoff[AL];
#pragma unroll
  for (int j = 0; j < AL; ++j) {
    const int f = min(wave + j * 4, AF - 1);      // row tile * 2 + half
    aoff[j] = (unsigned int)min((f >> 1) * 16 + col, p.M - 1) * p.lda +
              (f & 1) * 32 + hi * 8;
  }
  const bf16_t* wrow[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t)
    wrow[t] = p.W + (long long)min(n0 + t * 16 + col, p.N - 1) * p.K + hi * 8;

  u32x4_v ar[D][AL];
  bf16x8_v wr[D][CT][2];
  auto load_a = [&](int d, int s) {
    const bf16_t* a = p.A + (long long)min(s, s1 - 1) * 64;
#pragma unroll
    for (int j = 0; j < AL; ++j)
      ar[d][j] = *reinterpret_cast<const u32x4_v*>(a + aoff[j]);
  };
  auto load_w = [&](int d, int s) {
    const int k = min(s, s1 - 1) * 64;
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        wr[d][t][h] = *reinterpret_cast<const bf16x8_v*>(wrow[t] + k + h * 32);
  };
  auto store_a = [&](int d, int buf) {
#pragma unroll
    for (int j = 0; j < AL; ++j)
      if (AF % 4 == 0 || wave + j * 4 < AF)
        *reinterpret_cast<u32x4_v*>(
            &at[buf][(wave + j * 4) * 512 + lane * 8]) = ar[d][j];
  };
  f32x4_v acc[MT][CT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < CT; ++t) acc[m][t] = (f32x4_v){0.f, 0.f, 0.f, 0.f};

  // step s sits in place (s - s0) % D of the registers and half (s - s0) & 1
  // of LDS, which the step before last has left
#pragma unroll
  for (int d = 0; d < D; ++d) {
    load_a(d, s0 + d);
    load_w(d, s0 + d);
  }
  store_a(0, 0);
  load_a(0, s0 + D);
  lds_barrier();
  for (int sb = s0; sb < s1; sb += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int s = sb + d;
      store_a((d + 1) % D, (d + 1) & 1);
      load_a((d + 1) % D, s + 1 + D);
      // uniform; the loads take no branch, or their waits would meet there
      if (s < s1)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const bf16x8_v a = *reinterpret_cast<const bf16x8_v*>(
                &at[d & 1][(m * 2 + h) * 512 + lane * 8]);
#pragma unroll
            for (int t = 0; t < CT; ++t)
              acc[m][t] = mfma_bf16(wr[d][t][h], a, acc[m][t]);
          }
      load_w(d, s + D);
      lds_barrier();
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m * 16 + col;
    if (row >= p.M) continue;
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const int c = n0 + t * 16 + hi * 4;         // N % 16 == 0
      if (c < p.N)
        *reinterpret_cast<f32x4_v*>(
            p.part + ((long long)blockIdx.y * p.M + row) * p.N + c) =
            acc[m][t];
    }
  }
}

__global__ void __launch_bounds__(256)
qsa_rows_sum(const float* __restrict__ part, bf16_t* __restrict__ C,
             long long n, int S) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;                  // n % 4 == 0
  f32x4_v v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < S; ++s)
    v += *reinterpret_cast<const f32x4_v*>(part + s * n + i);
  *reinterpret_cast<uint2*>(C + i) =
      make_uint2(cvt_bf16x2(v[0], v[1]), cvt_bf16x2(v[2], v[3]));
}

// Shares of K: a block for each of the 256 CUs and none left over, which would
// have some CUs do the work of two (2560 x 10240 with 13 shares, 260 blocks:
// 28.8 us at 40 rows, 56.8 at 192; with 12: 19.5 and 34.7).
extern "C" int qsa_rows_gemm_shares(int N, int K) {
  const int blocks = (N + 127) / 128, steps = K >> 6;
  const int want = blocks < 256 ? 256 / blocks : 1;
  return want < steps ? want : steps;
}

extern "C" void qsa_rows_gemm_launch(const bf16_t* A, const bf16_t* W,
                                     bf16_t* C, float* part, int M, int N,
                                     int K, long long lda, int S,
                                     hipStream_t st) {
  const RowsArgs p{A, W, part, M, N, K, (unsigned int)lda};
  const dim3 grid((N + 127) / 128, S);
#define QSA_RG(MT) \
  hipLaunchKernelGGL((qsa_rows_gemm<MT>), grid, dim3(256), 0, st, p)
  if (M <= 48) QSA_RG(3);
  else if (M <= 64) QSA_RG(4);
  else if (M <= 96) QSA_RG(6);
  else if (M <= 128) QSA_RG(8);
  else QSA_RG(12);
#undef QSA_RG
  const long long n = (long long)M * N;
  hipLaunchKernelGGL(qsa_rows_sum, dim3((unsigned)((n / 4 + 255) / 256)),
                     dim3(256), 0, st, part, C, n, S);
}
