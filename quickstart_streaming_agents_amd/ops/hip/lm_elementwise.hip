// Row kernels of the mixer decoders: residual update + norm in f32, gated
// activation, latent norm + cache scatter, step slots, greedy pick.
#include "lm_common.h"

// ---------------------------------------------------------------------------
// Residual update and norm of one row, everything in f32:
//   r   = (init ? 0 : res) + p + tscale * table[ids[row]] + vec
//         (p, table, vec optional); p = y, or with POST the branch's own norm
//         y / sqrt(mean y^2 + eps) * post
//   res = r
//   out = norm(r) * w + b      LAYER: (r - mean)/sqrt(var + eps), var the
//                              mean squared deviation; else r/sqrt(mean r^2
//                              + eps).  b optional; without w, out = r.
// The row stays in registers between the passes up to CACHED groups per
// thread; wider rows re-read the residual this thread wrote itself.
// SHARES: y is a product whose shares of K have not been added; doing it here
// saves the launch that would (64 x 2048, four shares: 4.6 us).
// ---------------------------------------------------------------------------
template <typename T, int VEC, bool LAYER, bool POST, bool SHARES>
__global__ void __launch_bounds__(1024)
qsa_residual_norm(float* __restrict__ res, const T* __restrict__ y,
                  long long ystride, const float* __restrict__ parts,
                  long long pstep, int S, const T* __restrict__ post,
                  const T* __restrict__ table,
                  const long long* __restrict__ ids, float tscale,
                  const T* __restrict__ vec, const T* __restrict__ w,
                  const T* __restrict__ b, T* __restrict__ out, int W,
                  int vocab, float eps, int init) {
  constexpr int CACHED = 8;
  __shared__ float scratch[16];
  const long long row = blockIdx.x;
  float* rr = res + row * W;
  const T* yr = y ? y + row * ystride : nullptr;
  const T* er = nullptr;
  if (table) {
    long long id = ids[row];
    id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
    er = table + id * W;
  }
  auto load_y = [&](int i, float* v) {
    if constexpr (SHARES) ld_shares<VEC>(parts + row * W + i, pstep, S, v);
    else ldv<T, VEC>(yr + i, v);
  };
  const int step = blockDim.x * VEC;
  const int i0 = threadIdx.x * VEC;
  float cache[CACHED][VEC];
  float pinv = 1.f;
  if (POST) {
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < CACHED; ++c) {
      const int i = i0 + c * step;
      if (i < W) {
        load_y(i, cache[c]);
#pragma unroll
        for (int j = 0; j < VEC; ++j) ss = fmaf(cache[c][j], cache[c][j], ss);
      }
    }
    for (int i = i0 + CACHED * step; i < W; i += step) {
      float v[VEC];
      load_y(i, v);
#pragma unroll
      for (int j = 0; j < VEC; ++j) ss = fmaf(v[j], v[j], ss);
    }
    pinv = 1.f / sqrtf(block_reduce_sum(ss, scratch) / (float)W + eps);
  }
  float sum = 0.f;
  // v: on entry, with POST, the branch's output
  auto load_row = [&](int i, float* v) {
    float t[VEC];
    if (POST) {
      ldv<T, VEC>(post + i, t);
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[j] *= pinv * t[j];
      if (!init) {
        ldv<float, VEC>(rr + i, t);
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] += t[j];
      }
    } else {
      if (init) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = 0.f;
      } else {
        ldv<float, VEC>(rr + i, v);
      }
      if (SHARES || yr) {
        load_y(i, t);
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] += t[j];
      }
    }
    if (er) {
      ldv<T, VEC>(er + i, t);
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[j] = fmaf(tscale, t[j], v[j]);
    }
    if (vec) {
      ldv<T, VEC>(vec + i, t);
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[j] += t[j];
    }
    stv<float, VEC>(rr + i, v);
  };
#pragma unroll
  for (int c = 0; c < CACHED; ++c) {
    const int i = i0 + c * step;
    if (i < W) {
      load_row(i, cache[c]);
#pragma unroll
      for (int j = 0; j < VEC; ++j)
        sum += LAYER ? cache[c][j] : cache[c][j] * cache[c][j];
    }
  }
  for (int i = i0 + CACHED * step; i < W; i += step) {
    float v[VEC];
    if (POST) load_y(i, v);
    load_row(i, v);
#pragma unroll
    for (int j = 0; j < VEC; ++j) sum += LAYER ? v[j] : v[j] * v[j];
  }
  T* orow = out + row * W;
  if (!w) {                                         // the residual itself
#pragma unroll
    for (int c = 0; c < CACHED; ++c)
      if (i0 + c * step < W) stv<T, VEC>(orow + i0 + c * step, cache[c]);
    for (int i = i0 + CACHED * step; i < W; i += step) {
      float v[VEC];
      ldv<float, VEC>(rr + i, v);
      stv<T, VEC>(orow + i, v);
    }
    return;
  }
  sum = block_reduce_sum(sum, scratch);
  float mean = 0.f, ms = sum / (float)W;
  if (LAYER) {
    mean = ms;
    float dev = 0.f;
#pragma unroll
    for (int c = 0; c < CACHED; ++c)
      if (i0 + c * step < W) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          const float d = cache[c][j] - mean;
          dev = fmaf(d, d, dev);
        }
      }
    for (int i = i0 + CACHED * step; i < W; i += step) {
      float v[VEC];
      ldv<float, VEC>(rr + i, v);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float d = v[j] - mean;
        dev = fmaf(d, d, dev);
      }
    }
    ms = block_reduce_sum(dev, scratch) / (float)W;
  }
  const float inv = 1.f / sqrtf(ms + eps);
  auto emit = [&](int i, const float* v) {
    float t[VEC], o[VEC];
    ldv<T, VEC>(w + i, t);
#pragma unroll
    for (int j = 0; j < VEC; ++j) o[j] = (v[j] - mean) * inv * t[j];
    if (b) {
      ldv<T, VEC>(b + i, t);
#pragma unroll
      for (int j = 0; j < VEC; ++j) o[j] += t[j];
    }
    stv<T, VEC>(orow + i, o);
  };
#pragma unroll
  for (int c = 0; c < CACHED; ++c)
    if (i0 + c * step < W) emit(i0 + c * step, cache[c]);
  for (int i = i0 + CACHED * step; i < W; i += step) {
    float v[VEC];
    ldv<float, VEC>(rr + i, v);
    emit(i, v);
  }
}

// One group per thread: what a decoding step's few rows are.  Nothing but
// latency bounds these, so every load of the row goes out before the first one
// is waited for, what is absent (a null pointer) is read from the residual and
// not used, since a branch would wait for the loads ahead of it, and each sum
// has its own slots and so one barrier.  Sums and roundings are those of the
// kernel above, which its branches keep from being fused: a row has the same bits
// among 256 and among 257.  A 64-row step with 16 of them (2048 wide, shares of K)
// takes 641 us instead of 652, one row 345 instead of 354.
template <typename T, int VEC, bool LAYER, bool POST, bool SHARES>
__global__ void __launch_bounds__(1024)
qsa_residual_norm_once(float* __restrict__ res, const T* __restrict__ y,
                       long long ystride, const float* __restrict__ parts,
                       long long pstep, int S, const T* __restrict__ post,
                       const T* __restrict__ table,
                       const long long* __restrict__ ids, float tscale,
                       const T* __restrict__ vec, const T* __restrict__ w,
                       const T* __restrict__ b, T* __restrict__ out, int W,
                       int vocab, float eps, int init) {
  __shared__ float scratch[3][16];
  const long long row = blockIdx.x;
  const int i = threadIdx.x * VEC;
  const bool mine = i < W;
  const int at = mine ? i : W - VEC;
  const int waves = (W / VEC + 63) / 64;
  float* rr = res + row * W;
  const T* none = reinterpret_cast<const T*>(rr);
  const T* er = none;
  if (table) {
    long long id = ids[row];
    id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
    er = table + id * W;
  }
  float v[VEC], r[VEC], p[VEC], e[VEC], c[VEC], g[VEC], h[VEC];
  ldv<float, VEC>(rr + at, r);
  if constexpr (POST) ldv<T, VEC>(post + at, p);
  ldv<T, VEC>(er + at, e);
  ldv<T, VEC>((vec ? vec : none) + at, c);
  ldv<T, VEC>((w ? w : none) + at, g);
  ldv<T, VEC>((b ? b : none) + at, h);
  if constexpr (SHARES) ld_shares<VEC>(parts + row * W + at, pstep, S, v);
  else ldv<T, VEC>((y ? y + row * ystride : none) + at, v);
  __builtin_amdgcn_sched_barrier(0);

  auto block_sum = [&](float x, float* slots) {
    x = wave_reduce_sum(x);
    if ((threadIdx.x & 63) == 0) slots[threadIdx.x >> 6] = x;
    __syncthreads();
    float part[16], total = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) part[k] = slots[k];
#pragma unroll
    for (int k = 0; k < 16; ++k) total += k < waves ? part[k] : 0.f;
    return total;
  };
  if constexpr (POST) {
    float ss = 0.f;
    if (mine)
#pragma unroll
      for (int j = 0; j < VEC; ++j) ss = fmaf(v[j], v[j], ss);
    const float pinv =
        1.f / sqrtf(block_sum(ss, scratch[0]) / (float)W + eps);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
#pragma clang fp contract(off)
      v[j] *= pinv * p[j];
      if (!init) v[j] += r[j];
    }
  } else {
    const bool has = SHARES || y;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float x = init ? 0.f : r[j];
      v[j] = has ? x + v[j] : x;
    }
  }
  if (table)
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[j] = fmaf(tscale, e[j], v[j]);
  if (vec)
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[j] += c[j];
  if (mine) stv<float, VEC>(rr + i, v);
  T* orow = out + row * W;
  if (!w) {                                         // the residual itself
    if (mine) stv<T, VEC>(orow + i, v);
    return;
  }
  float sum = 0.f;
  if (mine)
#pragma unroll
    for (int j = 0; j < VEC; ++j) sum += LAYER ? v[j] : v[j] * v[j];
  sum = block_sum(sum, scratch[1]);
  float mean = 0.f, ms = sum / (float)W;
  if constexpr (LAYER) {
    mean = ms;
    float dev = 0.f;
    if (mine)
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float d = v[j] - mean;
        dev = fmaf(d, d, dev);
      }
    ms = block_sum(dev, scratch[2]) / (float)W;
  }
  const float inv = 1.f / sqrtf(ms + eps);
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
#pragma clang fp contract(off)
    v[j] = (v[j] - mean) * inv * g[j];
    if (b) v[j] += h[j];
  }
  if (mine) stv<T, VEC>(orow + i, v);
}

template <typename T, int VEC, bool LAYER, bool POST, bool SHARES>
static void residual_norm_go(float* res, const void* y, long long ystride,
                             const float* parts, int S,
                             const void* post, const void* table,
                             const long long* ids, float tscale,
                             const void* vec, const void* w, const void* b,
                             void* out, long long rows, int W, int vocab,
                             float eps, int init, hipStream_t st) {
  int threads = ((W + VEC - 1) / VEC + 63) / 64 * 64;
  // few rows: wide blocks, one round of loads; many rows: narrow ones
  const int most = rows <= 256 ? 1024 : 256;
  threads = threads > most ? most : threads;
  auto kernel = qsa_residual_norm<T, VEC, LAYER, POST, SHARES>;
  // Up to 256 rows a CU has one block at most and nothing hides its waits; with
  // more the other blocks do, and reading what is absent would be extra traffic.
  // us, above / so: steps of four layers 4096 wide, one row 450 / 446, 16 524 / 515,
  // 128 947 / 938, 200 1247 / 1225 (Lunulix), 336 / 333, 382 / 374, 665 / 655, 859 /
  // 850 (Luzalorn).  Launches alone, all of their operands in L2: layer norms of 1024 to
  // 4096 columns 2.8 to 5.8 / 2.3 to 4.9 for 1 to 256 rows, rms norms with a post norm
  // 3.0 to 5.6 / 2.4 to 5.0, those of shares 6.6 / 6.4 for 256 rows of 4096, but 3.3 /
  // 3.5 for one, whose absent operands are loads that no wait hides.
  if constexpr (VEC == 4) {
    if (rows <= 256 && W <= most * VEC)
      kernel = qsa_residual_norm_once<T, VEC, LAYER, POST, SHARES>;
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3(threads), 0, st, res,
                     (const T*)y, ystride, parts, rows * W, S,
                     (const T*)post, (const T*)table,
                     ids, tscale, (const T*)vec, (const T*)w, (const T*)b,
                     (T*)out, W, vocab, eps, init);
}

// parts and S: y as S shares [S][rows][W], bf16 storage and vec4 only
extern "C" void qsa_residual_norm_launch(
    float* res, const void* y, long long ystride, const float* parts, int S,
    const void* post,
    const void* table, const long long* ids, float tscale, const void* vec,
    const void* w, const void* b, void* out, long long rows, int W, int vocab,
    float eps, int init, int layer, int f32, int vec4, hipStream_t st) {
#define QSA_RN(T, V, L, P, H)                                                 \
  residual_norm_go<T, V, L, P, H>(res, y, ystride, parts, S, post, table,     \
                                  ids, tscale, vec, w, b, out, rows, W,       \
                                  vocab, eps, init, st)
#define QSA_RN_L(T, V, H)                                                     \
  if (layer) { if (post) QSA_RN(T, V, true, true, H);                         \
               else QSA_RN(T, V, true, false, H); }                           \
  else { if (post) QSA_RN(T, V, false, true, H);                              \
         else QSA_RN(T, V, false, false, H); }
  if (parts) {
    QSA_RN_L(bf16_t, 4, true)
  } else if (f32) {
    if (vec4) { QSA_RN_L(float, 4, false) } else { QSA_RN_L(float, 1, false) }
  } else {
    if (vec4) { QSA_RN_L(bf16_t, 4, false) } else { QSA_RN_L(bf16_t, 1, false) }
  }
#undef QSA_RN_L
#undef QSA_RN
}

// ---------------------------------------------------------------------------
// The Llama decoder's norm behind such a product: res <- res + sum of shares in
// bf16, out = rms norm of it times w, with the roundings of a stored product and
// of qsa_rmsnorm_kernel (elementwise.hip).  A row is one round of loads of its
// block (W <= 8192), S of them per thread.  192 x 4096, four shares: sum and norm
// as launches of their own 8.8 us, 5.2 here.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024)
qsa_rmsnorm_shares(const float* __restrict__ parts, long long step, int S,
                   bf16_t* __restrict__ res, const bf16_t* __restrict__ w,
                   bf16_t* __restrict__ out, int W, float eps) {
  __shared__ float scratch[16];
  const long long row = (long long)blockIdx.x * W;
  const int i = threadIdx.x * 8;
  float r[8], g[8], ss = 0.f;
  if (i < W) {
    float x[8];
    ldv<bf16_t, 8>(res + row + i, r);
    ldv<bf16_t, 8>(w + i, g);
    ld_shares<8>(parts + row + i, step, S, x);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      r[j] += x[j];
      ss = fmaf(r[j], r[j], ss);
      r[j] = bf16_to_f32(cvt_bf16(r[j]));
    }
    stv<bf16_t, 8>(res + row + i, r);
  }
  const float inv = rsqrtf(block_reduce_sum(ss, scratch) / (float)W + eps);
  if (i < W) {
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = r[j] * inv * g[j];
    stv<bf16_t, 8>(out + row + i, r);
  }
}

extern "C" void qsa_rmsnorm_shares_launch(const float* parts, int S,
                                          bf16_t* res, const bf16_t* w,
                                          bf16_t* out, long long rows, int W,
                                          float eps, hipStream_t st) {
  hipLaunchKernelGGL(qsa_rmsnorm_shares, dim3((unsigned)rows),
                     dim3((W / 8 + 63) / 64 * 64), 0, st, parts, rows * W, S,
                     res, w, out, W, eps);
}

// ---------------------------------------------------------------------------
// Gated activations.  The factor is the other half of a projection (a gated
// linear unit) or a slice of the token's row of a table:
//   out[r, c] = act(gate[r, c]) * up[r, c]
//   out[r, c] = act(gate[r, c]) * table[ids[r], col0 + c]
// act: silu, or the tanh form of gelu, z / (1 + exp(-2 sqrt(2/pi)
// (z + 0.044715 z^3))).
// ---------------------------------------------------------------------------
// S > 0 with a table: the gate is a product whose S shares have not been added.
template <typename T, int VEC, int ACT, bool SHARES>
__global__ void __launch_bounds__(256)
qsa_glu(const T* __restrict__ gate, const float* __restrict__ parts, int S,
        const T* __restrict__ up,
        const long long* __restrict__ ids, T* __restrict__ out,
        long long rows, long long cols, long long stride, long long ustride,
        long long vocab) {
  const long long groups = cols / VEC;
  const long long n = rows * groups;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const long long r = i / groups, c = (i % groups) * VEC;
    long long ur = r;
    if (ids) {
      ur = ids[r];
      ur = ur < 0 ? 0 : (ur >= vocab ? vocab - 1 : ur);
    }
    float g[VEC], u[VEC];
    if constexpr (SHARES) ld_shares<VEC>(parts + i * VEC, rows * cols, S, g);
    else ldv<T, VEC>(gate + r * stride + c, g);
    ldv<T, VEC>(up + ur * ustride + c, u);
#pragma unroll
    for (int j = 0; j < VEC; ++j)
      g[j] = act_f<sizeof(T) == 4, ACT>(g[j]) * u[j];
    stv<T, VEC>(out + r * cols + c, g);
  }
}

extern "C" void qsa_glu_launch(const void* gate, const float* parts, int S,
                               const void* up,
                               const long long* ids, void* out,
                               long long rows, long long cols,
                               long long stride, long long ustride,
                               long long vocab, int gelu, int f32, int vec,
                               hipStream_t st) {
  const long long n = rows * (cols / (vec ? 8 : 1));
  const long long want = (n + 255) / 256;
  dim3 grid((unsigned)(want < 1 ? 1 : (want > 16384 ? 16384 : want)));
#define QSA_GLU(T, V, A, H)                                                \
  hipLaunchKernelGGL((qsa_glu<T, V, A, H>), grid, dim3(256), 0, st,        \
                     (const T*)gate, parts, S, (const T*)up, ids, (T*)out, \
                     rows, cols, stride, ustride, vocab)
#define QSA_GLU_A(T, V, H)                                                 \
  if (gelu) QSA_GLU(T, V, QSA_ACT_GELU, H);                                \
  else QSA_GLU(T, V, QSA_ACT_SILU, H)
  if (parts) { QSA_GLU_A(bf16_t, 8, true); }
  else if (f32) {
    if (vec) { QSA_GLU_A(float, 8, false); }
    else { QSA_GLU_A(float, 1, false); }
  } else {
    if (vec) { QSA_GLU_A(bf16_t, 8, false); }
    else { QSA_GLU_A(bf16_t, 1, false); }
  }
#undef QSA_GLU_A
#undef QSA_GLU
}

// ---------------------------------------------------------------------------
// Latent norms of one projected row, both RMS with a plain weight:
//   blockIdx.y == 0: cq[row]        = rms(x[row, :qr]) * wq
//   blockIdx.y == 1: cache[slot]    = rms(x[row, qr:qr+kr]) * wk
// slot = page*64 + offset of the row's position; negative slots are skipped.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
qsa_latent_norm_store(const T* __restrict__ x, long long xstride,
                      const T* __restrict__ wq, const T* __restrict__ wk,
                      T* __restrict__ cq, T* __restrict__ cache,
                      const int* __restrict__ slots, int qr, int kr,
                      float eps) {
  __shared__ float scratch[8];
  const long long row = blockIdx.x;
  const bool lat = blockIdx.y == 1;
  const int n = lat ? kr : qr;
  const T* src = x + row * xstride + (lat ? qr : 0);
  const T* w = lat ? wk : wq;
  T* dst = cq + row * qr;
  if (lat) {
    const int slot = slots[row];
    if (slot < 0) return;                       // uniform over the block
    dst = cache + (long long)slot * kr;
  }
  float ss = 0.f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const float v = ldf<T>(src + i);
    ss = fmaf(v, v, ss);
  }
  ss = block_reduce_sum(ss, scratch);
  const float inv = 1.f / sqrtf(ss / (float)n + eps);
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    stf<T>(dst + i, ldf<T>(src + i) * inv * ldf<T>(w + i));
}

// The same with a wave per latent, which holds its row in registers and asks for
// all of it and the weights at once: bound by latency in a decoding step and by
// issue in a prompt.  13.8k rows of 768 + 512: two-byte loads, twice, 38.9 us,
// 16.3 here; one row 3.7 and 2.9.
template <typename T>
__global__ void __launch_bounds__(256)
qsa_latent_norm_wave(const T* __restrict__ x, long long xstride,
                     const T* __restrict__ wq, const T* __restrict__ wk,
                     T* __restrict__ cq, T* __restrict__ cache,
                     const int* __restrict__ slots, long long rows, int qr,
                     int kr, float eps) {
  constexpr int G = 4;                              // groups of 4 per lane
  const long long unit = (long long)blockIdx.x * 4 +
                         __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long row = unit >> 1;
  if (row >= rows) return;
  const bool lat = unit & 1;
  const int n = lat ? kr : qr;
  const int i = (threadIdx.x & 63) * 4;
  const T* src = x + row * xstride + (lat ? qr : 0);
  const T* w = lat ? wk : wq;
  const int slot = slots[row];
  float v[G][4], g[G][4];
#pragma unroll
  for (int c = 0; c < G; ++c) ldv<T, 4>(src + min(i + c * 256, n - 4), v[c]);
#pragma unroll
  for (int c = 0; c < G; ++c) ldv<T, 4>(w + min(i + c * 256, n - 4), g[c]);
  __builtin_amdgcn_sched_barrier(0);
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < G; ++c)
    if (i + c * 256 < n)
#pragma unroll
      for (int j = 0; j < 4; ++j) ss = fmaf(v[c][j], v[c][j], ss);
  const float inv = 1.f / sqrtf(wave_reduce_sum(ss) / (float)n + eps);
  if (lat && slot < 0) return;
  T* dst = lat ? cache + (long long)slot * kr : cq + row * qr;
#pragma unroll
  for (int c = 0; c < G; ++c)
    if (i + c * 256 < n) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[c][j] *= inv * g[c][j];
      stv<T, 4>(dst + i + c * 256, v[c]);
    }
}

extern "C" void qsa_latent_norm_store_launch(
    const void* x, long long xstride, const void* wq, const void* wk,
    void* cq, void* cache, const int* slots, long long rows, int qr, int kr,
    float eps, int f32, hipStream_t st) {
  // a wave per latent where groups of 4 divide and align everything and a wave
  // holds the widest; other rows go element by element
  const int size = f32 ? 4 : 2;
  auto whole = [&](const void* p) { return ((size_t)p & (4 * size - 1)) == 0; };
  if (qr >= 4 && kr >= 4 && qr <= 1024 && kr <= 1024 && qr % 4 == 0 &&
      kr % 4 == 0 && xstride % 4 == 0 && whole(x) && whole(wq) && whole(wk) &&
      whole(cq) && whole(cache)) {
    dim3 waves((unsigned)((rows + 1) / 2));
    if (f32)
      hipLaunchKernelGGL((qsa_latent_norm_wave<float>), waves, dim3(256), 0,
                         st, (const float*)x, xstride, (const float*)wq,
                         (const float*)wk, (float*)cq, (float*)cache, slots,
                         rows, qr, kr, eps);
    else
      hipLaunchKernelGGL((qsa_latent_norm_wave<bf16_t>), waves, dim3(256), 0,
                         st, (const bf16_t*)x, xstride, (const bf16_t*)wq,
                         (const bf16_t*)wk, (bf16_t*)cq, (bf16_t*)cache,
                         slots, rows, qr, kr, eps);
    return;
  }
  dim3 grid((unsigned)rows, 2);
  if (f32)
    hipLaunchKernelGGL((qsa_latent_norm_store<float>), grid, dim3(256), 0, st,
                       (const float*)x, xstride, (const float*)wq,
                       (const float*)wk, (float*)cq, (float*)cache, slots, qr,
                       kr, eps);
  else
    hipLaunchKernelGGL((qsa_latent_norm_store<bf16_t>), grid, dim3(256), 0,
                       st, (const bf16_t*)x, xstride, (const bf16_t*)wq,
                       (const bf16_t*)wk, (bf16_t*)cq, (bf16_t*)cache, slots,
                       qr, kr, eps);
}

// ---------------------------------------------------------------------------
// Cache slot of every decode row's newest position (-1: row not in use).
// ---------------------------------------------------------------------------
__global__ void qsa_decode_slots(const int* __restrict__ block_table,
                                 const int* __restrict__ seq_lens,
                                 int* __restrict__ slots, int B,
                                 int max_pages) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  const int p = seq_lens[b] - 1;
  slots[b] = (p < 0 || p / 64 >= max_pages)
                 ? -1
                 : block_table[(long long)b * max_pages + p / 64] * 64 +
                       p % 64;
}

extern "C" void qsa_decode_slots_launch(const int* block_table,
                                        const int* seq_lens, int* slots,
                                        int B, int max_pages,
                                        hipStream_t st) {
  hipLaunchKernelGGL(qsa_decode_slots, dim3((B + 63) / 64), dim3(64), 0, st,
                     block_table, seq_lens, slots, B, max_pages);
}

// ---------------------------------------------------------------------------
// Greedy pick: index of the largest logit of each row, the lowest index on
// ties.  One block per row and no scratch memory to clear, so it can be
// recorded into a graph.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(1024)
qsa_argmax_rows(const T* __restrict__ x, long long* __restrict__ out, int n) {
  __shared__ float sv[16];
  __shared__ int si[16];
  const T* r = x + (long long)blockIdx.x * n;
  float best = -INFINITY;
  int at = 0x7fffffff;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const float v = ldf<T>(r + i);
    if (v > best || at == 0x7fffffff) { best = v; at = i; }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float v = __shfl_xor(best, off, QSA_WAVE);
    const int i = __shfl_xor(at, off, QSA_WAVE);
    if (v > best || (v == best && i < at)) { best = v; at = i; }
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sv[wave] = best; si[wave] = at; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k)
      if (sv[k] > best || (sv[k] == best && si[k] < at)) {
        best = sv[k];
        at = si[k];
      }
    out[blockIdx.x] = at < n ? at : 0;
  }
}

extern "C" void qsa_argmax_rows_launch(const void* x, long long* out,
                                       long long rows, int n, int f32,
                                       hipStream_t st) {
  if (f32)
    hipLaunchKernelGGL((qsa_argmax_rows<float>), dim3((unsigned)rows),
                       dim3(1024), 0, st, (const float*)x, out, n);
  else
    hipLaunchKernelGGL((qsa_argmax_rows<bf16_t>), dim3((unsigned)rows),
                       dim3(1024), 0, st, (const bf16_t*)x, out, n);
}
