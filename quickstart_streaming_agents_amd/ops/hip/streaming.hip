// Streaming-analytics kernels: batched windowed aggregation (K7) and the
// batched per-key AR anomaly scorer (K3).
#include <algorithm>

#include "common.h"

// ---------------------------------------------------------------------------
// Windowed aggregation: segmented count/sum by (key, window) over an event
// batch.  window = (ts - t0) / win_ms; out slot = key * nwin + window.
// The reference shape: TUMBLE(...) GROUP BY key (LAB3:99-133, LAB4:127-141).
//
// Bound by atomics, not bytes: those of different dies meet behind the L2s, at
// some 12 G/s whether they collide or not (two per event: 334 us for 2M
// events, 1000 keys of uneven weight, 288 windows).  So blocks count chunks of
// consecutive events, which in a stream span a few windows, in LDS, and a chunk
// whose span does not fit goes to the output event by event.  How the cells of
// a chunk reach the output is chosen by qsa_window_workspace:
//   merged   chunks of 4096 leave (windows spanned) * nkeys cells in a
//            workspace, qsa_window_merge adds them up, without atomics and in
//            a fixed order (26 us, clearing the output and both launches)
//   direct   chunks of 256 or 1024 add their cells to the output with atomics
// More keys than fit in LDS have neither: an event at a time.
// ---------------------------------------------------------------------------
#define QSA_AGG_CELLS 6144             // 48 KiB of LDS: three blocks per CU
#define QSA_AGG_FEW 2048               // of a chunk of 256: more cost more to
                                       // clear and look through than to miss
#define QSA_AGG_CHUNK 4096
#define QSA_AGG_BLOCKS 2048            // most chunks, 96 MiB of workspace

__device__ __forceinline__ int qsa_window_of(long long ts, long long t0,
                                             long long win_ms, int nwin) {
  const long long w = (ts - t0) / win_ms;
  return w >= 0 && w < nwin ? (int)w : -1;
}

// The same for win_ms > 0 without a 64-bit division (some 130 instructions):
// a quotient below 2^31 from the reciprocal is off by one at most.
// limit = nwin * win_ms, inv = 1 / win_ms.
__device__ __forceinline__ int qsa_window_by(long long ts, long long t0,
                                             long long win_ms, long long limit,
                                             double inv) {
  const long long d = ts - t0;
  if (d <= -win_ms || d >= limit) return -1;
  int w = (int)((double)d * inv);
  const long long r = d - w * win_ms;
  w += r >= win_ms ? 1 : r < 0 ? -1 : 0;
  return max(w, 0);                    // the quotient is cut towards zero
}

// A launch of its own: up to 100k events are bound by the host, for whom a tensor's
// fill is dearer (an aggregation 10.2 us with it, 9.2 so; 2M events 23.1 both). The
// grid is bounded, since a launch holds fewer than 2^32 threads: tables of more than
// 268 MB take several turns of it.
#define QSA_CLEAR_BLOCKS 65536
__global__ void __launch_bounds__(256)
qsa_window_clear(int* __restrict__ cells, long long n) {
  const long long step = (long long)gridDim.x * 1024;
  for (long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4; i < n; i += step)
    if (i + 4 <= n)
      *reinterpret_cast<int4*>(cells + i) = make_int4(0, 0, 0, 0);
    else
      for (long long j = i; j < n; ++j) cells[j] = 0;
}

// An event at a time, straight to the output.
__global__ void __launch_bounds__(256)
qsa_window_events(const long long* __restrict__ ts,
                  const int* __restrict__ key,
                  const float* __restrict__ value,  // nullptr -> count only
                  int* __restrict__ counts, float* __restrict__ sums,
                  long long t0, long long win_ms, int nwin, int nkeys,
                  long long n) {
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  for (; i < n; i += (long long)gridDim.x * 256) {
    const int w = qsa_window_of(ts[i], t0, win_ms, nwin), k = key[i];
    if (w < 0 || k < 0 || k >= nkeys) continue;
    const long long slot = (long long)k * nwin + w;
    atomicAdd(counts + slot, 1);
    if (value) unsafeAtomicAdd(sums + slot, value[i]);
  }
}

// A value as a whole number of units of 2^unit; exact where its lowest bit is no
// less than one (see the kernel).
struct QsaBits {
  unsigned mant;                       // 24 bits, 0: the value is zero
  int exp;                             // of the mantissa's lowest bit
};

__device__ __forceinline__ QsaBits qsa_bits(float v) {
  const unsigned u = __float_as_uint(v), e = u >> 23 & 255, f = u & 0x7fffff;
  return {e ? f | 0x800000 : f, (int)max(e, 1u) - 150};
}

__device__ __forceinline__ long long qsa_units(float v, int unit) {
  const QsaBits b = qsa_bits(v);
  const int s = b.exp - unit;          // below 0: zeros are shifted out
  const long long x = b.mant == 0 ? 0
                      : s >= 0    ? (long long)b.mant << s
                                  : (long long)(b.mant >> -s);
  return v < 0.f ? -x : x;
}

// The least of a wave, by exchanges between registers: through LDS the ranges of
// windows and of values were 24 of them one behind another, of which those of the
// values cost counts and sums of values that do not fit 2 to 6 % of their time (2M
// events, 7 keys: counts 16.4 us without them, 17.2 with, 16.2 so; wide values
// 27.9, 28.9 and 28.4; 1M events, 20 keys, 19.5, 20.6 and 20.3).
template <int CTRL, int ROWS>
__device__ __forceinline__ int qsa_dpp_min(int v) {
  return min(v, __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ int qsa_wave_min(int v) {
  v = qsa_dpp_min<0x111, 0xf>(v);      // from 1, 2, 4, 8 lanes below in a row
  v = qsa_dpp_min<0x112, 0xf>(v);
  v = qsa_dpp_min<0x114, 0xf>(v);
  v = qsa_dpp_min<0x118, 0xf>(v);
  v = qsa_dpp_min<0x142, 0xa>(v);      // a row's last to the odd row above
  v = qsa_dpp_min<0x143, 0xc>(v);      // lane 31 to the upper two rows
  return __builtin_amdgcn_readlane(v, 63);
}

// A float added to LDS occupies the unit some 3 cycles a lane, a 64-bit integer
// under a third of that: of 20 us for 2M events of 1000 keys 10 were these sums
// (7 so, with 512 threads a chunk, 256 before).  So where
// the values of a chunk allow it their sums are whole numbers of the lowest bit
// that is set in any of them, in one word with the count: exact, in any order,
// rounded once at the end.  They do if the highest is below 2^38 of these units
// (as 24-bit numbers do within 2^14 of each other), for 4096 of them then stay
// below the 2^50 that the word has room for.  Others, and chunks of more, are
// float sums.
#define QSA_AGG_SUM_BITS 51
#define QSA_AGG_UNIT_BITS 38

// PER events of a thread, chunk == NT * PER; PER 0: any.  win_ms > 0.
template <int PER, int CELLS, int NT>
__global__ void __launch_bounds__(NT)
qsa_window_agg(const long long* __restrict__ ts, const int* __restrict__ key,
               const float* __restrict__ value,  // nullptr -> count only
               int* __restrict__ counts, float* __restrict__ sums,
               long long t0, long long win_ms, int nwin, int nkeys,
               long long n, long long chunk,
               int2* __restrict__ span,          // [blocks] {first, windows}
               int* __restrict__ ws) {           // [blocks, 2, QSA_AGG_CELLS]
  constexpr bool FIT = PER > 4;        // smaller chunks gain nothing by it
  static_assert(!FIT || (long long)PER * NT <= 1 << (QSA_AGG_SUM_BITS - 1 -
                                             QSA_AGG_UNIT_BITS) &&
                            (long long)PER * NT <
                                1 << (64 - QSA_AGG_SUM_BITS),
                "the sum and the count of a chunk fit");
  __shared__ unsigned long long cell[CELLS];     // or counts, then float sums
  __shared__ int lo_s, hi_s, bit_s, top_s;
  int* cnt = reinterpret_cast<int*>(cell);
  float* sum = reinterpret_cast<float*>(cell) + CELLS;
  const int tid = threadIdx.x;
  const long long first = (long long)blockIdx.x * chunk;
  const long long end = min(first + chunk, n);
  if (tid == 0) {
    lo_s = bit_s = 0x7fffffff;
    hi_s = -1;
    top_s = -0x7fffffff;
  }
  __syncthreads();
  int lo = 0x7fffffff, hi = -1;
  int bit = 0x7fffffff, top = -0x7fffffff;       // lowest bit, highest 24 bits
  // PER: every load of the chunk is under way before the first is used, and
  // an event's window is found once
  int win[PER ? PER : 1], ek[PER ? PER : 1];
  float ev[PER ? PER : 1];
  if constexpr (PER > 0) {
    long long et[PER];
    const long long limit = win_ms > 0x7fffffffffffffffll / nwin
                                ? 0x7fffffffffffffffll : win_ms * nwin;
    const double inv = 1.0 / (double)win_ms;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const long long i = min(first + tid + j * NT, n - 1);
      et[j] = ts[i];
      ek[j] = key[i];
      ev[j] = value ? value[i] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      win[j] = first + tid + j * NT < end
                   ? qsa_window_by(et[j], t0, win_ms, limit, inv) : -1;
      if (win[j] >= 0) {
        lo = min(lo, win[j]);
        hi = max(hi, win[j]);
        if (FIT && value) {
          const QsaBits b = qsa_bits(ev[j]);
          if (b.mant && ek[j] >= 0 && ek[j] < nkeys) {
            bit = min(bit, b.exp + __ffs(b.mant) - 1);
            top = max(top, b.exp);     // 255 - 150: not a number, infinite
          }
        }
      }
    }
  } else {
#pragma unroll 4
    for (long long i = first + tid; i < end; i += NT) {
      const int w = qsa_window_of(ts[i], t0, win_ms, nwin);
      if (w >= 0) {
        lo = min(lo, w);
        hi = max(hi, w);
      }
    }
  }
  lo = qsa_wave_min(lo);
  hi = ~qsa_wave_min(~hi);
  if (FIT && value) {
    bit = qsa_wave_min(bit);
    top = ~qsa_wave_min(~top);
  }
  if ((tid & 63) == 0) {
    atomicMin(&lo_s, lo);
    atomicMax(&hi_s, hi);
    if (FIT && value) {
      atomicMin(&bit_s, bit);
      atomicMax(&top_s, top);
    }
  }
  __syncthreads();
  lo = lo_s;
  hi = hi_s;
  const long long cells = hi < 0 ? 0 : (long long)(hi - lo + 1) * nkeys;
  const bool local = cells <= CELLS;     // uniform over the block, as is whole
  if (ws && tid == 0)
    span[blockIdx.x] = make_int2(lo, local && hi >= 0 ? hi - lo + 1 : 0);
  if (cells == 0) return;              // no event of the chunk counts
  int unit = 0;                        // no value but zeros: any
  bool whole = false;
  if constexpr (FIT) {
    const bool some = bit_s != 0x7fffffff;
    if (some) unit = bit_s;
    whole = local && value &&
            (!some || (top_s < 255 - 150 &&
                       top_s + 24 - bit_s <= QSA_AGG_UNIT_BITS));
  }
  if (local) {
    for (int c = tid; c < (int)cells; c += NT) {
      if (whole) {
        cell[c] = 0;
      } else {
        cnt[c] = 0;
        sum[c] = 0.f;
      }
    }
    __syncthreads();
  }
  auto count = [&](int w, int kk, float v) {
    if (w < 0 || kk < 0 || kk >= nkeys) return;
    if (local) {
      const int c = (w - lo) * nkeys + kk;
      if (whole) {
        atomicAdd(cell + c, (1ull << QSA_AGG_SUM_BITS) +
                                (unsigned long long)qsa_units(v, unit));
        return;
      }
      atomicAdd(cnt + c, 1);
      if (value) unsafeAtomicAdd(sum + c, v);
    } else {
      const long long slot = (long long)kk * nwin + w;
      atomicAdd(counts + slot, 1);
      if (value) unsafeAtomicAdd(sums + slot, v);
    }
  };
  if constexpr (PER > 0) {
#pragma unroll
    for (int j = 0; j < PER; ++j) count(win[j], ek[j], ev[j]);
  } else {
#pragma unroll 4
    for (long long i = first + tid; i < end; i += NT)
      count(qsa_window_of(ts[i], t0, win_ms, nwin), key[i],
            value ? value[i] : 0.f);
  }
  if (!local) return;
  __syncthreads();
  const double one = __longlong_as_double((long long)(unit + 1023) << 52);
  for (int c = tid; c < (int)cells; c += NT) {
    int many;
    float v;
    if (whole) {
      constexpr int UP = 64 - QSA_AGG_SUM_BITS;
      const long long word = (long long)cell[c], x = word << UP >> UP;
      many = (int)((unsigned long long)(word - x) >> QSA_AGG_SUM_BITS);
      v = (float)((double)x * one);
    } else {
      many = cnt[c];
      v = sum[c];
    }
    if (ws) {
      int* wc = ws + (long long)blockIdx.x * 2 * QSA_AGG_CELLS + c;
      wc[0] = many;
      if (value) wc[QSA_AGG_CELLS] = __float_as_int(v);
    } else if (many) {
      const long long slot = (long long)(c % nkeys) * nwin + lo + c / nkeys;
      atomicAdd(counts + slot, many);
      if (value) unsafeAtomicAdd(sums + slot, v);
    }
  }
}

// Block = 8 windows x 64 keys, a wave per window: the chunks that reach it, in
// order, added to what other chunks left in the output.  Bound by a chain of
// latencies (spans, cells, output), so the output is fetched first and four
// chunks' cells at a time; the output is read and written with 8 windows of a
// key in neighbouring lanes, where a wave's 64 keys were 64 lines, four times:
// 288 x 1000 cells of 489 chunks 12 us before, 9 so.
__global__ void __launch_bounds__(512)
qsa_window_merge(const int2* __restrict__ span, const int* __restrict__ ws,
                 int blocks, int* __restrict__ counts,
                 float* __restrict__ sums, int has_value, int nwin,
                 int nkeys) {
  __shared__ int list[QSA_AGG_BLOCKS];
  __shared__ int2 range[QSA_AGG_BLOCKS];
  __shared__ int wave_n[8];
  __shared__ int out_c[8][65];
  __shared__ float out_v[8][65];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w0 = blockIdx.x * 8, w = w0 + wave, k0 = blockIdx.y * 64;
  const int k = k0 + lane;
  const bool live = k < nkeys && w < nwin;
  // a thread's cell of the output: 8 windows of a key are 8 lanes, one line
  const int ow = tid & 7, ok = tid >> 3;
  const bool mine = k0 + ok < nkeys && w0 + ow < nwin;
  const long long slot = mine ? (long long)(k0 + ok) * nwin + w0 + ow : 0;
  const int c = counts[slot];
  const float v = has_value ? sums[slot] : 0.f;
  int total = 0;
  for (int base = 0; base < blocks; base += 512) {
    const int b = base + tid;
    const int2 s = b < blocks ? span[b] : make_int2(0, 0);
    const bool in = s.y > 0 && s.x < w0 + 8 && s.x + s.y > w0;
    const unsigned long long m = __ballot(in);
    if (lane == 0) wave_n[wave] = __popcll(m);
    __syncthreads();
    int at = total + __popcll(m & ((1ull << lane) - 1));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i < wave) at += wave_n[i];
      total += wave_n[i];
    }
    if (in) {
      list[at] = b;
      range[at] = s;
    }
    __syncthreads();
  }
  // in a stream most groups do not reach this window
  int pc = 0;
  float pv = 0.f;
  bool reached = false;
  for (int j0 = 0; j0 < total; j0 += 4) {
    bool any = false, in[4];
    int at[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      at[j] = min(j0 + j, total - 1);
      const int2 s = range[at[j]];
      in[j] = j0 + j < total && w >= s.x && w < s.x + s.y;
      any |= in[j];
    }
    if (!any) continue;                // uniform over the wave
    reached = true;
    int gc[4];
    float gv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      gc[j] = 0;
      gv[j] = 0.f;
      if (in[j] && live) {
        const int* p = ws + (long long)list[at[j]] * 2 * QSA_AGG_CELLS +
                       (w - range[at[j]].x) * nkeys + k;
        gc[j] = *p;
        if (has_value) gv[j] = __int_as_float(p[QSA_AGG_CELLS]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      pc += gc[j];
      pv += gv[j];
    }
  }
  out_c[wave][lane] = pc;
  out_v[wave][lane] = pv;
  if (lane == 0) wave_n[wave] = reached;
  __syncthreads();
  if (mine && wave_n[ow]) {
    counts[slot] = c + out_c[ow][ok];
    if (has_value) sums[slot] = v + out_v[ow][ok];
  }
}

// ---------------------------------------------------------------------------
// Batched AR(p)+ridge anomaly scorer: one wave (64 lanes) per key series.
// Mirrors runtime/anomaly.py ar_forecast(): centered lag design, ridge
// lambda = 0.3 * tr(G)/p, prediction se with leverage.  p <= 4.
// series: [K, Tmax] f32 (ragged via lengths[]); outputs per key.
//
// Bound by latency: three passes over a series.  All lanes share every pass and
// solve the padded 4x4 system in registers (rows beyond p are the identity).
// A series of up to 512 goes to LDS at once, beside its length: passes that
// waited for memory 64 numbers at a time made 10.5 us of 1000 series of 288,
// 8.9 so (171 us with the solve and the residuals on one lane).  Many short ones
// keep LDS busy as it is, with the sums over lanes: 30,000 of 128 43.3 us read
// from memory, 45.8 from LDS, 8000 16.3 both, 4000 11.2 and 11.0; 30,000 of 150
// 50.4 and 48.1.
// ---------------------------------------------------------------------------
#define QSA_AR_MAXP 4

template <int STAGE>                   // Tmax <= STAGE, or 0: any
__global__ void __launch_bounds__(64)
qsa_anomaly_batch(const float* __restrict__ series, const int* __restrict__ lengths,
                  float* __restrict__ forecast, float* __restrict__ pred_se,
                  int* __restrict__ dof_out, int Tmax, int order) {
  const int kidx = blockIdx.x;
  const int lane = threadIdx.x;
  const float* row = series + (long long)kidx * Tmax;
  const int n = lengths[kidx];
  __shared__ float staged[STAGE ? STAGE : 1];
  const float* h;
  if constexpr (STAGE > 0) {           // without waiting for the length
    float x[STAGE / QSA_WAVE];
#pragma unroll
    for (int j = 0; j < STAGE / QSA_WAVE; ++j)
      if (j * QSA_WAVE < Tmax) x[j] = row[min(lane + j * QSA_WAVE, Tmax - 1)];
#pragma unroll
    for (int j = 0; j < STAGE / QSA_WAVE; ++j)
      if (j * QSA_WAVE < Tmax) staged[lane + j * QSA_WAVE] = x[j];
    __syncthreads();
    h = staged;
  } else {
    h = row;
  }

  if (n < 6) {  // mean/std fallback (matches CPU path)
    float sum = 0.f, sq = 0.f;
    for (int i = lane; i < n; i += QSA_WAVE) {
      sum += h[i];
      sq = fmaf(h[i], h[i], sq);
    }
    sum = wave_reduce_sum(sum);
    sq = wave_reduce_sum(sq);
    if (lane == 0) {
      const float mean = n > 0 ? sum / n : 0.f;
      float sd = n > 1 ? sqrtf(fmaxf((sq - n * mean * mean) / (n - 1), 0.f))
                       : fabsf(mean) + 1.f;
      forecast[kidx] = mean;
      pred_se[kidx] = fmaxf(sd, 1e-9f);
      dof_out[kidx] = max(n - 1, 1);
    }
    return;
  }

  int p = min(order, max(1, (n - 4) / 4));
  p = min(p, QSA_AR_MAXP);
  const int m = n - p;

  // accumulate: colsum[j] (lag j+1), ysum, then centered cross products.
  float colsum[QSA_AR_MAXP + 1];  // [0] = y
#pragma unroll
  for (int j = 0; j <= QSA_AR_MAXP; ++j) colsum[j] = 0.f;
  for (int t = p + lane; t < n; t += QSA_WAVE) {
    colsum[0] += h[t];
#pragma unroll
    for (int j = 1; j <= QSA_AR_MAXP; ++j)
      if (j <= p) colsum[j] += h[t - j];
  }
#pragma unroll
  for (int j = 0; j <= QSA_AR_MAXP; ++j) colsum[j] = wave_reduce_sum(colsum[j]);
  const float ym = colsum[0] / m;
  float xm[QSA_AR_MAXP];
#pragma unroll
  for (int j = 0; j < QSA_AR_MAXP; ++j) xm[j] = (j < p) ? colsum[j + 1] / m : 0.f;

  // G = Xc'Xc (p x p), b = Xc'yc
  float G[QSA_AR_MAXP][QSA_AR_MAXP], bb[QSA_AR_MAXP];
#pragma unroll
  for (int a = 0; a < QSA_AR_MAXP; ++a) {
    bb[a] = 0.f;
#pragma unroll
    for (int c = 0; c < QSA_AR_MAXP; ++c) G[a][c] = 0.f;
  }
  for (int t = p + lane; t < n; t += QSA_WAVE) {
    float xc[QSA_AR_MAXP];
#pragma unroll
    for (int j = 0; j < QSA_AR_MAXP; ++j)
      xc[j] = (j < p) ? h[t - 1 - j] - xm[j] : 0.f;
    const float yc = h[t] - ym;
#pragma unroll
    for (int a = 0; a < QSA_AR_MAXP; ++a) {
      bb[a] = fmaf(xc[a], yc, bb[a]);
#pragma unroll
      for (int c = 0; c < QSA_AR_MAXP; ++c)
        G[a][c] = fmaf(xc[a], xc[c], G[a][c]);
    }
  }
#pragma unroll
  for (int a = 0; a < QSA_AR_MAXP; ++a) {
    bb[a] = wave_reduce_sum(bb[a]);
#pragma unroll
    for (int c = 0; c < QSA_AR_MAXP; ++c)         // symmetric, to the last bit
      G[a][c] = c < a ? G[c][a] : wave_reduce_sum(G[a][c]);
  }

  // ridge solve (G + lam I) [coef | y] = [b | x_next] by Gauss-Jordan, every
  // lane the same; x_next' y is the leverage of the newest lags
  float tr = 0.f;
#pragma unroll
  for (int a = 0; a < QSA_AR_MAXP; ++a) tr += G[a][a];   // 0 beyond p
  const float lam = 0.3f * (tr / p + 1e-12f);
  constexpr int W = QSA_AR_MAXP + 2;
  float A[QSA_AR_MAXP][W], xn[QSA_AR_MAXP];
#pragma unroll
  for (int a = 0; a < QSA_AR_MAXP; ++a) {
    xn[a] = a < p ? h[n - 1 - a] - xm[a] : 0.f;
#pragma unroll
    for (int c = 0; c < QSA_AR_MAXP; ++c)
      A[a][c] = G[a][c] + (a == c ? (a < p ? lam : 1.f) : 0.f);
    A[a][QSA_AR_MAXP] = bb[a];
    A[a][QSA_AR_MAXP + 1] = xn[a];
  }
#pragma unroll
  for (int col = 0; col < QSA_AR_MAXP; ++col) {
#pragma unroll
    for (int row = col + 1; row < QSA_AR_MAXP; ++row) {
      const bool swap = fabsf(A[row][col]) > fabsf(A[col][col]);
#pragma unroll
      for (int c = 0; c < W; ++c) {
        const float u = A[col][c], v = A[row][c];
        A[col][c] = swap ? v : u;
        A[row][c] = swap ? u : v;
      }
    }
    const float d = A[col][col];
    const float dinv = (fabsf(d) > 1e-30f) ? 1.f / d : 0.f;
#pragma unroll
    for (int c = 0; c < W; ++c) A[col][c] *= dinv;
#pragma unroll
    for (int row = 0; row < QSA_AR_MAXP; ++row) {
      if (row == col) continue;
      const float f = A[row][col];
#pragma unroll
      for (int c = 0; c < W; ++c) A[row][c] -= f * A[col][c];
    }
  }
  float rr = 0.f;                      // residual sum of squares
#pragma unroll 4
  for (int t = p + lane; t < n; t += QSA_WAVE) {
    float pred = 0.f;
#pragma unroll
    for (int j = 0; j < QSA_AR_MAXP; ++j)
      if (j < p) pred = fmaf(A[j][QSA_AR_MAXP], h[t - 1 - j] - xm[j], pred);
    const float r = h[t] - ym - pred;
    rr = fmaf(r, r, rr);
  }
  rr = wave_reduce_sum(rr);
  if (lane == 0) {
    const int dof = max(m - (p + 1), 1);
    const float resid_var = rr / dof;
    float fc = ym, lever = 1.f / m;
#pragma unroll
    for (int j = 0; j < QSA_AR_MAXP; ++j) {
      fc = fmaf(A[j][QSA_AR_MAXP], xn[j], fc);
      lever = fmaf(A[j][QSA_AR_MAXP + 1], xn[j], lever);
    }
    forecast[kidx] = fc;
    pred_se[kidx] =
        fmaxf(sqrtf(fmaxf(resid_var, 1e-18f) * (1.f + fmaxf(lever, 0.f))),
              1e-9f);
    dof_out[kidx] = dof;
  }
}

extern "C" long long qsa_window_chunk(long long n) {
  return std::max<long long>(
      QSA_AGG_CHUNK, (n + QSA_AGG_BLOCKS - 1) / QSA_AGG_BLOCKS);
}

// Words of workspace, 0 for the direct form.  Merging costs a second launch and
// a pass over the output, 18 us for the smallest, so it takes 64 chunks (in
// order, 400 keys, 288 windows, direct / merged: 200k events 17 / 21 us, 300k
// 21 / 21, 500k 28 / 21), and it pays only where chunks fit in LDS.  In a stream
// a chunk spans 4096 nwin / n windows and touches up to one more; where six in
// ten would touch more than fit, or no chunk can, the direct form is ahead
// (1000 keys, 288 windows, 200k events: 21 us against 40; 3000, 500k: 44 / 79;
// 6000, 1M: 94 / 128; but 3000, 1M: 81 / 50 and 6000, 2M: 169 / 169).  Events in
// no order have the merge in vain (7 us), except where the whole table fits:
// there 17 chunks are enough (20 keys, 300 windows, 200k events: in order 8.6 /
// 18, in none 62 / 29).
extern "C" long long qsa_window_workspace(long long n, long long nkeys,
                                          long long nwin, long long win_ms) {
  const long long chunk = qsa_window_chunk(n), blocks = (n + chunk - 1) / chunk;
  if (win_ms <= 0 || nkeys <= 0) return 0;
  const long long fit = QSA_AGG_CELLS / nkeys;   // windows
  if (fit == 0 || blocks <= (nwin <= fit ? 16 : 64) ||
      10.0 * chunk * nwin > (double)n * (10 * fit - 4))
    return 0;
  return blocks * (2 + 2 * QSA_AGG_CELLS);
}

extern "C" void qsa_window_clear_launch(int* cells, long long n,
                                        hipStream_t stream) {
  if (n > 0) {
    const long long blocks = (n + 1023) / 1024;
    hipLaunchKernelGGL(qsa_window_clear,
                       dim3((unsigned)(blocks < QSA_CLEAR_BLOCKS ? blocks
                                                                 : QSA_CLEAR_BLOCKS)),
                       dim3(256), 0, stream, cells, n);
  }
}

extern "C" void qsa_window_agg_launch(const long long* ts, const int* key,
                                      const float* value, int* counts,
                                      float* sums, long long t0,
                                      long long win_ms, int nwin, int nkeys,
                                      long long n, int* ws,
                                      hipStream_t stream) {
  if (n == 0 || nwin <= 0 || nkeys <= 0) return;
  if (win_ms <= 0 || nkeys > QSA_AGG_CELLS) {
    // 4096 blocks at most: 7000 keys, 8M events 832 us, 976 with a block for
    // every 256
    const unsigned grid =
        (unsigned)std::min<long long>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(qsa_window_events, dim3(grid), dim3(256), 0, stream, ts,
                       key, value, counts, sums, t0, win_ms, nwin, nkeys, n);
    return;
  }
  // direct: chunks of 256 until they give every CU two blocks (1000 keys, 288
  // windows, 100k events: 15.0 us, 15.8 with chunks of 1024; 200k: 22.7, 20.9)
  const long long chunk = ws ? qsa_window_chunk(n)
                             : n <= 512 * 256 ? 256 : 1024;
  const int blocks = (int)((n + chunk - 1) / chunk);
  int2* span = reinterpret_cast<int2*>(ws);
  int* cells = ws ? ws + 2 * blocks : nullptr;
#define QSA_AGG(PER, CELLS, NT)                                              \
  hipLaunchKernelGGL((qsa_window_agg<PER, CELLS, NT>), dim3(blocks),         \
                     dim3(NT), 0, stream, ts, key, value, counts, sums, t0,  \
                     win_ms, nwin, nkeys, n, chunk, span, cells)
  if (chunk > QSA_AGG_CHUNK) QSA_AGG(0, QSA_AGG_CELLS, 256);
  else if (ws) QSA_AGG(QSA_AGG_CHUNK / 512, QSA_AGG_CELLS, 512);
  else if (chunk == 1024) QSA_AGG(4, QSA_AGG_CELLS, 256);
  else QSA_AGG(1, QSA_AGG_FEW, 256);
#undef QSA_AGG
  if (ws)
    hipLaunchKernelGGL(qsa_window_merge,
                       dim3((nwin + 7) / 8, (nkeys + 63) / 64), dim3(512), 0,
                       stream, span, cells, blocks, counts, sums,
                       value ? 1 : 0, nwin, nkeys);
}

extern "C" void qsa_anomaly_batch_launch(const float* series,
                                         const int* lengths, float* forecast,
                                         float* pred_se, int* dof_out, int K,
                                         int Tmax, int order,
                                         hipStream_t stream) {
  if (Tmax <= 512 && (Tmax > 2 * QSA_WAVE || K <= 8192))
    hipLaunchKernelGGL(qsa_anomaly_batch<512>, dim3(K), dim3(64), 0, stream,
                       series, lengths, forecast, pred_se, dof_out, Tmax,
                       order);
  else
    hipLaunchKernelGGL(qsa_anomaly_batch<0>, dim3(K), dim3(64), 0, stream,
                       series, lengths, forecast, pred_se, dof_out, Tmax,
                       order);
}
