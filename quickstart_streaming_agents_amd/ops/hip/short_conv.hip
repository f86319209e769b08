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

template <typename T, int VEC>
__global__ void __launch_bounds__(256) qsa_conv_qkv(ConvQkv p) {
  conv_qkv_unit<T, VEC>(p, blockIdx.x, blockIdx.y * blockDim.x + threadIdx.x,
                        blockIdx.z, gridDim.z);
}

extern "C" void qsa_conv_qkv_launch(ConvQkv p, int chunks, int f32, int vec4,
                                    hipStream_t st) {
  const int V = vec4 ? 4 : 1;
  const int units = conv_qkv_units(p, V);
  const int threads = units <= 64 ? 64 : units <= 128 ? 128 : 256;
  const int across = (units + threads - 1) / threads;
  const dim3 grid((unsigned)chunks, (unsigned)across,
                  (unsigned)conv_parts(p.step, p.taps, (long long)chunks * across));
#define QSA_CQ(T, V) \
  hipLaunchKernelGGL((qsa_conv_qkv<T, V>), grid, dim3(threads), 0, st, p)
  if (f32) { if (vec4) QSA_CQ(float, 4); else QSA_CQ(float, 1); }
  else     { if (vec4) QSA_CQ(bf16_t, 4); else QSA_CQ(bf16_t, 1); }
#undef QSA_CQ
}

template <typename T, int VEC>
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
                                     int chunks, void* out, int C, int f32,
                                     int vec4, hipStream_t st) {
  const int units = vec4 ? C / 4 : C;
  const int threads = units <= 64 ? 64 : units <= 128 ? 128 : 256;
  const int across = (units + threads - 1) / threads;
  const dim3 grid((unsigned)chunks, (unsigned)across,
                  (unsigned)conv_parts(step, taps, (long long)chunks * across));
#define QSA_CS(T, V)                                                        \
  hipLaunchKernelGGL((qsa_conv_silu<T, V>), grid, dim3(threads), 0, st,     \
                     (const T*)x, xstride, w, bias, taps, (T*)tails, step,  \
                     (T*)out, C)
  if (f32) { if (vec4) QSA_CS(float, 4); else QSA_CS(float, 1); }
  else     { if (vec4) QSA_CS(bf16_t, 4); else QSA_CS(bf16_t, 1); }
#undef QSA_CS
}
