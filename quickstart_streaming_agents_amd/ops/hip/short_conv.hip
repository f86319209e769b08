// Short causal convolutions over time, one filter per channel:
//   y_t[c] = bias[c] + sum_j w[j][c] u_(t - taps + 1 + j)[c]
// u are columns of a projected row; zeros stand before a sequence's first
// token, and the last taps - 1 inputs of every sequence are its tail:
// tails [slots, taps - 1, C] in the storage type, oldest first.
//
// A thread owns a few channels for CONV_ROWS tokens of one portion (its window
// stays in registers).  Only the first tokens of a portion look at the old
// tail, and the thread that owns them also writes the new one, so reading and
// writing it never race.  Tail entries before position 0 read as zero: slots
// need no clearing between owners.
//
//   qsa_conv_qkv   channels [q | k | v] of an attention layer, then the
//                  rotation of q and k; k and v go straight to their pages
//   qsa_conv_silu  bias and silu, to a dense [rows, C]
#include "short_conv.h"

// Parts of a chunk's rows: blocks that leave CUs idle are latencies one behind another,
// so several share a chunk (us: 60 tokens of 4096 channels to pages / with silu 9.9 /
// 6.6 -> 6.3 / 5.0, 900 11.3 / 7.5 -> 8.5 / 6.9, but 1800, 226 blocks, 13.3 / 10.7 ->
// 15.0 / 11.2).
static int conv_parts(const ConvStep& st, int taps, long long blocks) {
  return st.item && taps - 1 <= CONV_ROWS / CONV_PARTS && blocks <= 128 ? CONV_PARTS
                                                                       : 1;
}

// Whether tokens go one by one.  Where there are more waves than fit the chip at once
// with the registers of many tokens ahead, eight a CU, fewer registers are more in
// flight.  us, tokens ahead / one by one, to pages, 4096 channels with four taps: 3600
// tokens, 1824 waves, 18.9 / 21.7, 4000 in portions of 40, 2400 waves, 23.3 / 21.5, 5000
// 26.5 / 25.0, 7500 32.3 / 28.8, 14,000 58.3 / 54.7; of 768 channels 14,000 tokens, 1750
// waves, 14.8 / 16.5.  With silu there are registers for either: 7500 33.8 / 40.2.  And
// where portions have two or three tokens there is little to be ahead of: 60 of two, of
// 174, 768 and 4096 channels, to pages 4.0, 4.3, 4.7 / 3.6, 4.0, 4.4, with silu 3.4, 3.5,
// 3.8 / 3.0, 3.3, 3.6; 40 of five 4.6, 5.1, 5.6 / 4.3, 5.3, 5.6.
static bool conv_single(const ConvStep& st, long long rows, int chunks,
                        long long waves) {
  return st.item && (rows < 4ll * chunks || waves > 2048);
}

template <typename T, int VEC, bool SINGLE>
__global__ void __launch_bounds__(256) qsa_conv_qkv(ConvQkv p) {
  conv_qkv_unit<T, VEC, false, SINGLE>(p, blockIdx.x,
                                       blockIdx.y * blockDim.x + threadIdx.x,
                                       blockIdx.z, gridDim.z);
}

extern "C" void qsa_conv_qkv_launch(ConvQkv p, long long rows, int chunks,
                                    int f32, int vec4, hipStream_t st) {
  const int V = vec4 ? 4 : 1;
  const int units = conv_qkv_units(p, V);
  const int threads = units <= 64 ? 64 : units <= 128 ? 128 : 256;
  const int across = (units + threads - 1) / threads;
  const long long blocks = (long long)chunks * across;
  const bool single = conv_single(p.step, rows, chunks, blocks * (threads / 64));
  const dim3 grid((unsigned)chunks, (unsigned)across,
                  single ? 1u : (unsigned)conv_parts(p.step, p.taps, blocks));
#define QSA_CQ(T, V)                                                         \
  if (single)                                                                \
    hipLaunchKernelGGL((qsa_conv_qkv<T, V, true>), grid, dim3(threads), 0,   \
                       st, p);                                               \
  else                                                                       \
    hipLaunchKernelGGL((qsa_conv_qkv<T, V, false>), grid, dim3(threads), 0,  \
                       st, p)
  if (f32) { if (vec4) { QSA_CQ(float, 4); } else { QSA_CQ(float, 1); } }
  else     { if (vec4) { QSA_CQ(bf16_t, 4); } else { QSA_CQ(bf16_t, 1); } }
#undef QSA_CQ
}

template <typename T, int VEC, bool SINGLE>
__global__ void __launch_bounds__(256)
qsa_conv_silu(const T* x, long long xstride, const float* __restrict__ w,
              const float* __restrict__ bias, int taps, T* tails,
              ConvStep step, T* __restrict__ out, int C) {
  const int u = blockIdx.y * blockDim.x + threadIdx.x;
  if (u >= C / VEC) return;
  const ConvSpan s = conv_span(step, blockIdx.x, blockIdx.z, gridDim.z);
  if (s.slot < 0 || s.p0 < 0 || s.t0 >= s.n) return;
  T* tail = tails + (long long)s.slot * (taps - 1) * C;
  const int c0 = u * VEC, c1 = c0;
  auto pre = [](int) { return 0; };
  auto emit = [=](int t, float (&a)[1][VEC], int) {
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      a[0][i] = sizeof(T) == 4 ? silu_f(a[0][i])
                               : a[0][i] / (1.f + __expf(-a[0][i]));
    stv<T, VEC>(out + (long long)(s.r0 + t) * C + c0, a[0]);
  };
  CONV_DISPATCH(T, VEC, 1)
}

extern "C" void qsa_conv_silu_launch(const void* x, long long xstride,
                                     const float* w, const float* bias,
                                     int taps, void* tails, ConvStep step,
                                     long long rows, int chunks, void* out,
                                     int C, int f32, int vec4, hipStream_t st) {
  const int units = vec4 ? C / 4 : C;
  const int threads = units <= 64 ? 64 : units <= 128 ? 128 : 256;
  const int across = (units + threads - 1) / threads;
  const long long blocks = (long long)chunks * across;
  const bool single = conv_single(step, rows, chunks, 0);
  const dim3 grid((unsigned)chunks, (unsigned)across,
                  single ? 1u : (unsigned)conv_parts(step, taps, blocks));
#define QSA_CS_AS(T, V, SINGLE)                                              \
  hipLaunchKernelGGL((qsa_conv_silu<T, V, SINGLE>), grid, dim3(threads), 0,  \
                     st, (const T*)x, xstride, w, bias, taps, (T*)tails,     \
                     step, (T*)out, C)
#define QSA_CS(T, V)                                                         \
  if (single) QSA_CS_AS(T, V, true); else QSA_CS_AS(T, V, false)
  if (f32) { if (vec4) { QSA_CS(float, 4); } else { QSA_CS(float, 1); } }
  else     { if (vec4) { QSA_CS(bf16_t, 4); } else { QSA_CS(bf16_t, 1); } }
#undef QSA_CS
#undef QSA_CS_AS
}
