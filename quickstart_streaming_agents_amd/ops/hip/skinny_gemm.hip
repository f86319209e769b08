// Skinny-batch decode GEMM for CDNA4 (gfx950): C[M,N] = A[M,K] @ W[N,K]^T,
// M <= 32 (the decode batch), bf16 in / bf16 out.
// Serves the decode projections of the agents' language models.
//
// Decode projections are HBM-bandwidth-bound on the WEIGHT stream (the
// activations are KB-sized): speed-of-light is W bytes / 6.3 TB/s.  rocBLAS
// general-GEMM tiles for big M and loses on the latency-critical small
// shapes at M~24.  The kernel is skinny_stream.h's.
//
// W is packed once at model init into [N/16, K/32, 16, 32]: one wave
// instruction reads one 1 KiB 16x32 fragment block.
//
// Whether W is read past the last-level cache (skinny_stream.h, FAR) is the caller's
// to say, who knows what else a step reads; matrices below 4 MB stay there.
// Block shapes follow the fp8 form's measurements: one tile of 16 columns per
// block, two from 6144 columns on; 4 waves for K up to 2048, 8 above.
#include "skinny_stream.h"

template <int WAVES, int TILES, int MT, bool FAR>
__global__ void __launch_bounds__(WAVES * 64)
qsa_skinny_gemm(SkinnyArgs p) {
  skinny_stream<WAVES, TILES, MT, false, ROWS, false, false, false, FAR>(p);
}

template <int WAVES, int TILES>
static void bf16_go(const SkinnyArgs& p, hipStream_t st) {
  const dim3 grid(p.N / (16 * TILES)), block(WAVES * 64);
#define QSA_GO(MT, FAR)                                                      \
  hipLaunchKernelGGL((qsa_skinny_gemm<WAVES, TILES, MT, FAR>), grid, block,  \
                     0, st, p)
  if (p.M <= 16) {
    if (p.far) QSA_GO(1, true); else QSA_GO(1, false);
  } else {
    if (p.far) QSA_GO(2, true); else QSA_GO(2, false);
  }
#undef QSA_GO
}

static SkinnyArgs bf16_args(const unsigned short* A, const unsigned short* Wf,
                            unsigned short* C, int M, int N, long long K,
                            long long lda, bool far) {
  return SkinnyArgs{A, reinterpret_cast<const u32x4_v*>(Wf), nullptr, C,
                    nullptr, nullptr, nullptr, nullptr, M, N, 0, K, lda,
                    0.f, far && (long long)N * K >= 2 << 20};
}

extern "C" void qsa_skinny_gemm_launch(const unsigned short* A,
                                       const unsigned short* Wf,
                                       unsigned short* Cbf, int M, int N,
                                       long long K, long long lda, bool far,
                                       hipStream_t stream) {
  const SkinnyArgs p = bf16_args(A, Wf, Cbf, M, N, K, lda, far);
  if (K <= 2048) bf16_go<4, 1>(p, stream);
  else if (N >= 6144 && N % 32 == 0) bf16_go<8, 2>(p, stream);
  else bf16_go<8, 1>(p, stream);
}

// Tuning probe of tools/kernel_bench.py: any block shape.
extern "C" int qsa_skinny_gemm_probe_launch(
    const unsigned short* A, const unsigned short* Wf, unsigned short* Cbf,
    int M, int N, long long K, long long lda, int waves, int tiles,
    hipStream_t stream) {
  const SkinnyArgs p = bf16_args(A, Wf, Cbf, M, N, K, lda, true);
#define QSA_CASE(W, T)               \
  if (waves == W && tiles == T) {    \
    bf16_go<W, T>(p, stream);        \
    return 1;                        \
  }
  QSA_CASE(4, 1) QSA_CASE(8, 1) QSA_CASE(16, 1) QSA_CASE(4, 2) QSA_CASE(8, 2)
#undef QSA_CASE
  return 0;
}
