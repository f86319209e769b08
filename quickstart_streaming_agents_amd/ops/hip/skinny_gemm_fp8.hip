// FP8 (OCP e4m3) weight-streaming decode GEMM for CDNA4 (gfx950):
// C[M,N] = A[M,K] @ (s[N] * Q[N,K])^T, M <= 32, A bf16, Q fp8, C bf16.
// Serves the decode projections of the agents' language models.
//
// The bf16 skinny kernel (skinny_gemm.hip) is HBM-bound on the WEIGHT
// stream (PMC: ~3% MFMA util); its ceiling is W bytes / 6.3 TB/s.  FP8
// weights HALVE that stream: per-output-channel symmetric quantization
// (s[n] = max|W[n,:]| / 448, the standard W8A16 weight-only scheme) keeps
// activations bf16 and applies the scale once in the epilogue — zero
// inner-loop cost.  Dequant in-kernel: v_cvt_scalef32_pk_bf16_fp8 with a scale of
// one (2 fp8 -> 2 bf16).  It is exact: e4m3 has 3 mantissa bits, bf16 has 8, and
// every e4m3 value (normals and denormals) is a bf16 value, so the MFMA math
// matches a bf16 kernel running on the dequantized weights.
//
// The kernel is skinny_stream.h's, with the norms, activation and residual of a
// decoding step done on the way.
//
// Pack layout [N/16, K/64, 16, 4, 2, 8] ("fragment-pair-major"): one lane
// reads ONE 16-byte vector covering its 8 fp8 for TWO consecutive
// 16x16x32 k-fragments -> full-width dwordx4 loads on a byte stream.
// Gfx950 also has native fp8 MFMA, but using it would force the
// ACTIVATIONS to fp8 too (non-scaled fp8 MFMA is A8W8); this kernel is
// bandwidth-bound, so bf16 MFMA at half the weight bytes is the same
// speed with better numerics.
#include "skinny_stream.h"

template <int WAVES, int TILES, int MT, int FORM, bool NORM, bool GLU,
          bool RES, bool FAR>
__global__ void __launch_bounds__(WAVES * 64)
qsa_skinny_gemm_fp8(SkinnyArgs p) {
  skinny_stream<WAVES, TILES, MT, true, FORM, NORM, GLU, RES, FAR>(p);
}

template <int WAVES, int FORM, bool FAR>
__global__ void __launch_bounds__(WAVES * 64)
qsa_skinny_gemm_fp8_half(SkinnyArgs p) {
  skinny_stream<WAVES, 1, 1, true, FORM, false, false, true, FAR, true>(p);
}

template <int WAVES, int TILES, bool NORM, bool GLU, bool RES>
static void fp8_go(const SkinnyArgs& p, int pack, hipStream_t st) {
  const dim3 grid(p.N / (16 * TILES)), block(WAVES * 64);
#define QSA_GO_AS(MT, FORM, FAR)                                              \
  hipLaunchKernelGGL(                                                         \
      (qsa_skinny_gemm_fp8<WAVES, TILES, MT, FORM, NORM, GLU, RES, FAR>),     \
      grid, block, 0, st, p)
#define QSA_GO(MT, FORM)                                                      \
  if (p.far) QSA_GO_AS(MT, FORM, true); else QSA_GO_AS(MT, FORM, false)
  if (p.M <= FEW && !pack) {
    QSA_GO(1, FEW_ROWS);
  } else if (p.M <= 16) {
    if (pack) { QSA_GO(1, PACKED); } else { QSA_GO(1, ROWS); }
  } else {
    if (pack) { QSA_GO(2, PACKED); } else { QSA_GO(2, ROWS); }
  }
#undef QSA_GO
#undef QSA_GO_AS
}

// Blocks, measured on the projections of 2048- and 4096-wide decoders: waves
// get at least 8 steps of K each, so 4 of them share K up to 2048 and 8 above;
// two tiles of columns as soon as 192 blocks are left (half the A reads per
// weight).  Four tiles for a vocabulary, and from 16384 columns on where A is
// two row tiles and costs more than the weights (28672 x 4096, 32 rows: 37 us
// with two tiles, 29 with four).
// With 9 to 16 rows A still is twice the weights, and four tiles of K beyond 2048 are
// ahead from 24577 columns on where the CU with most blocks has no more tiles so than in
// blocks of two: up to 32768, from 40961 to 49152 and 57345 to 65536 (us with two / four:
// 25600 x 3072 18.7 / 16.8, 32768 21.1 / 19.2, but 24576 16.6 / 16.9, 36864 24.0 / 24.3
// and of K 4096 29.5 / 32.2; 49152 x 5120 47.0 / 42.6; 61440 x 4096 45.4 / 43.3; of 160
// shapes of K 2304 to 8192 the choice is 0.2 % from the best, at most 5 %).
// 12288 to 16384 columns are one block of four tiles for a CU, and with eight waves (us
// at 16 / 24 rows, eight waves of two tiles -> so: 12288 x 2048 7.9 / 9.9 -> 7.4 / 7.8;
// 16384 x 3072 11.3 / 14.3 -> 10.6 / 11.3; of 24 rows 12288 x 1024 8.7 -> 5.6, 15360 x
// 4096 17.4 -> 14.4; but of 16 13.9 -> 15.0, and 16384 x 4096 with 24 rows 16.2 in four
// waves of four, 16.8 so).
// us at 1 / 16 rows, one tile per block and row-major A before -> here (packed
// from 5 rows on, norm or residual included): 6144 x 4096 13.1 / 14.2 -> 7.5 /
// 8.6; 4096 x 4096 8.1 / 9.4 -> 6.2 / 7.2; 28672 x 4096 32 / 36 -> 24.6 / 27.9
// with the gating; 4096 x 14336 22 / 25 -> 14.7 / 17.9; 128256 x 2048 57 / 62
// -> 48.6 / 52.2 (5.4 TB/s).
extern "C" void qsa_skinny_fp8_block(int M, int N, long long K, int glu, int res,
                                     int* waves, int* tiles) {
  const bool whole = N % (glu ? 128 : 64) == 0 && M > (glu ? 8 : 0) && !res;
  const bool once = M > 8 && N >= 12288 && N <= 16384 &&
                    (M > 16 ? K >= 1024 && (K != 4096 || N < 16384)
                            : K >= 2048 && K <= 3072);
  // tiles of the CU with most blocks, in blocks of four and of two
  const bool even = (N + 16383) / 16384 * 4 == (N + 8191) / 8192 * 2;
  const bool four = N >= 65536 || (M > 16 && N >= 16384) ||
                    (M > 8 && K > 2048 && N > 24576 && even);
  if (whole && (once || four)) {
    *waves = once ? 8 : 4;
    *tiles = 4;
  } else if (glu) {
    *waves = K <= 2048 ? 4 : 8;
    *tiles = 2;
  } else {
    *tiles = N >= 6144 && N % 32 == 0 ? 2 : 1;
    *waves = *tiles == 1 && K <= 2048 ? 4 : 8;
  }
}

template <bool NORM, bool GLU, bool RES>
static void fp8_any(const SkinnyArgs& p, int pack, hipStream_t st) {
  int waves, tiles;
  qsa_skinny_fp8_block(p.M, p.N, p.K, GLU, RES, &waves, &tiles);
  if constexpr (!RES)
    if (tiles == 4)
      return waves == 8 ? fp8_go<8, 4, NORM, GLU, RES>(p, pack, st)
                        : fp8_go<4, 4, NORM, GLU, RES>(p, pack, st);
  if constexpr (GLU) {
    if (waves == 4) fp8_go<4, 2, NORM, GLU, RES>(p, pack, st);
    else fp8_go<8, 2, NORM, GLU, RES>(p, pack, st);
  } else {
    if (tiles == 2) fp8_go<8, 2, NORM, GLU, RES>(p, pack, st);
    else if (waves == 4) fp8_go<4, 1, NORM, GLU, RES>(p, pack, st);
    else fp8_go<8, 1, NORM, GLU, RES>(p, pack, st);
  }
}

// Whether a product with a residual is done in half tiles: up to 2048 columns are
// 128 tiles or fewer, and from 3072 numbers of K on a block's part of the stream is
// more than it has in flight at once (us at 1 / 4 / 8 rows, weights from memory, whole
// tiles -> half ones: 2048 x 8192 8.0 / 8.6 / 9.7 -> 5.6 / 6.3 / 6.2; 2048 x 4096 5.1 /
// 5.3 / 6.0 -> 4.2 / 4.6 / 4.6; 1024 x 3072 4.6 / 5.0 / 5.3 -> 3.7 / 4.2 / 4.1; 512 x
// 14336 10.7 / 12.0 / 14.0 -> 7.5 / 9.4 / 8.6; but 2048 x 2048 3.8 / 4.1 / 4.3 -> 3.7 /
// 4.2 / 4.1, 2560 x 8192 9.1 / 8.9 / 10.0 -> 8.2 / 9.8 / 9.6).  16 layers of width 2048,
// a step of one row 517 -> 495 us, of eight 570 -> 536; 8 layers, 4 rows 308 -> 293.
extern "C" int qsa_skinny_fp8_half(int M, int N, long long K) {
  return M <= 8 && N <= 2048 && K >= 3072 && K % 128 == 0;
}

static void fp8_half(const SkinnyArgs& p, int pack, hipStream_t st) {
  const dim3 grid(p.N / 8);
#define QSA_HALF_AS(WAVES, FORM, FAR)                                         \
  hipLaunchKernelGGL((qsa_skinny_gemm_fp8_half<WAVES, FORM, FAR>), grid,      \
                     dim3(WAVES * 64), 0, st, p)
#define QSA_HALF(WAVES, FORM)                                                 \
  if (p.far) QSA_HALF_AS(WAVES, FORM, true);                                  \
  else QSA_HALF_AS(WAVES, FORM, false)
#define QSA_HALF_OF(WAVES)                                                    \
  if (pack) { QSA_HALF(WAVES, PACKED); }                                      \
  else if (p.M <= FEW) { QSA_HALF(WAVES, FEW_ROWS); }                         \
  else { QSA_HALF(WAVES, ROWS); }
  if (p.K < 6144) {                    // a wave has 6 or more steps
    QSA_HALF_OF(4)
  } else {
    QSA_HALF_OF(8)
  }
#undef QSA_HALF_OF
#undef QSA_HALF
#undef QSA_HALF_AS
}

extern "C" void qsa_skinny_gemm_fp8_launch(
    const unsigned short* A, const unsigned char* Qf, const float* scale,
    unsigned short* C, unsigned short* next, int M, int N, long long K,
    long long lda, int pack, const unsigned short* norm_w, const float* ss_in,
    int parts, float eps, int glu, float* ss_out, int far, hipStream_t stream) {
  const SkinnyArgs p{A, reinterpret_cast<const u32x4_v*>(Qf), scale, C, next,
                     norm_w, ss_in, ss_out, M, N, parts, K, lda, eps,
                     far != 0};
  if (ss_out && qsa_skinny_fp8_half(M, N, K)) fp8_half(p, pack, stream);
  else if (ss_out) fp8_any<false, false, true>(p, pack, stream);
  else if (ss_in && glu) fp8_any<true, true, false>(p, pack, stream);
  else if (ss_in) fp8_any<true, false, false>(p, pack, stream);
  else fp8_any<false, false, false>(p, pack, stream);
}

// Tuning probe of tools/fp8_bench.py: plain form, any block shape.
extern "C" int qsa_skinny_gemm_fp8_probe_launch(
    const unsigned short* A, const unsigned char* Qf, const float* scale,
    unsigned short* C, int M, int N, long long K, long long lda, int pack,
    int waves, int tiles, hipStream_t stream) {
  const SkinnyArgs p{A, reinterpret_cast<const u32x4_v*>(Qf), scale, C,
                     nullptr, nullptr, nullptr, nullptr, M, N, 0, K, lda,
                     0.f, true};
#define QSA_CASE(W, T)                                      \
  if (waves == W && tiles == T) {                           \
    fp8_go<W, T, false, false, false>(p, pack, stream);     \
    return 1;                                               \
  }
  QSA_CASE(4, 1) QSA_CASE(8, 1) QSA_CASE(4, 2) QSA_CASE(8, 2) QSA_CASE(4, 4)
  QSA_CASE(8, 4)
#undef QSA_CASE
  return 0;
}

// First rows of a step: res <- embed[tokens], the operand of the projection
// that norms them, and their sums of squares as one part.
__global__ void __launch_bounds__(256)
qsa_embed_rows(const bf16_t* __restrict__ embed,
               const long long* __restrict__ tokens,
               const bf16_t* __restrict__ w, bf16_t* __restrict__ res,
               bf16_t* __restrict__ next, float* __restrict__ ss, int H,
               long long vocab, int mt) {
  __shared__ float scratch[4];
  const int row = blockIdx.x;
  const long long tok = tokens[row];
  const bool ok = tok >= 0 && tok < vocab;
  const u32x4_v* src = reinterpret_cast<const u32x4_v*>(
      embed + (ok ? tok : 0) * H);
  float s = 0.f;
  for (int i = threadIdx.x; i < H / 8; i += 256) {
    // a token that the table does not have gives no number, not another row
    const u32x4_v v = ok ? src[i] : (u32x4_v)(0x7fc07fc0u);
    const u32x4_v g = reinterpret_cast<const u32x4_v*>(w)[i];
    u32x4_v o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float2 f = bf16x2_to_f32x2(v[e]), u = bf16x2_to_f32x2(g[e]);
      s = fmaf(f.x, f.x, fmaf(f.y, f.y, s));
      o[e] = cvt_bf16x2(f.x * u.x, f.y * u.y);
    }
    *reinterpret_cast<u32x4_v*>(res + (long long)row * H + i * 8) = v;
    *reinterpret_cast<u32x4_v*>(
        next + (mt ? packed_at(row, i * 8, mt) : (long long)row * H + i * 8)) =
        o;
  }
  s = block_reduce_sum(s, scratch);
  if (threadIdx.x == 0) ss[row * 4] = s;
}

extern "C" void qsa_embed_rows_launch(const unsigned short* embed,
                                      const long long* tokens,
                                      const unsigned short* w,
                                      unsigned short* res,
                                      unsigned short* next, float* ss, int M,
                                      int H, long long vocab, int mt,
                                      hipStream_t stream) {
  hipLaunchKernelGGL(qsa_embed_rows, dim3(M), dim3(256), 0, stream, embed,
                     tokens, w, res, next, ss, H, vocab, mt);
}
