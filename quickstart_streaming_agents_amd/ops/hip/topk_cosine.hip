// HBM-resident vector search: exact cosine top-k (the K2 hot op).
//
// Replaces the reference's MongoDB Atlas $vectorSearch (lab2 main.tf:215:
// 1536-dim cosine, k=3, numCandidates=500) with an exact scan of the
// normalized index matrix in HBM.
//
// Bound by one read of the index.  A block scores 16*T documents against 16*QT
// queries at once on the f32 matrix cores (16x16x4, f32 products and sums), so
// up to 16 queries cost one read of the matrix; its four waves split the vector
// dimension and meet in LDS, so small indexes still spread over the chip.  T = 4
// keeps 8 KiB of documents per wave on their way while the previous step
// multiplies; T = 1 serves indexes whose 64-document blocks would leave CUs idle.
// 100,000 x 1536, k = 3: 8 queries 146 us with rows loaded straight into the
// matrix cores' layout, 112 through LDS, 98 past the last-level cache (6.3 TB/s),
// and 7 of merge; 32 queries 200 and 136; 10,000 documents, 8 queries 19.5 and 14.7.
//
// Results: scores > -2 in descending order, equal scores by ascending
// document; what k asks for beyond them is (-2, -1).  NaN scores never enter.
#include "common.h"


using f32x4_t = __attribute__((ext_vector_type(4))) float;

__device__ __forceinline__ bool qsa_better(float s, int i, float t, int j) {
  return s > t || (s == t && i < j);
}

// The best k of a block's 16*T documents for each of its queries, from its four
// waves' sums; `part` is [4][16*T][17].
template <int T, int QT>
__device__ __forceinline__ void qsa_topk_candidates(
    float (*part)[16 * T][17], const double (&total)[T][QT][4], int doc0,
    int q0, float* __restrict__ cand_scores, int* __restrict__ cand_ids, int Qn,
    int N, int k) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, hi = lane >> 4;
#pragma unroll
  for (int u = 0; u < QT; ++u) {       // 16 queries at a time
    if (u) __syncthreads();
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[wave][t * 16 + hi * 4 + r][col] = (float)total[t][u][r];
    __syncthreads();
    // 16 lanes per query, T documents each: k rounds of best-of-the-rest
    const int q = tid >> 4, sub = tid & 15, qi = q0 + u * 16 + q;
    float sc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int d = t * 16 + sub;
      const float v = (float)(((double)part[0][d][q] + part[1][d][q]) +
                              ((double)part[2][d][q] + part[3][d][q]));
      sc[t] = doc0 + d < N && v > -2.0f ? v : -INFINITY;
    }
    const bool live = qi < Qn;
    const long long at =
        ((long long)qi * gridDim.x + blockIdx.x) * k;
    for (int r = 0; r < k; ++r) {
      float bs = sc[0];
      int bi = doc0 + sub;
#pragma unroll
      for (int t = 1; t < T; ++t)
        if (sc[t] > bs) {
          bs = sc[t];
          bi = doc0 + t * 16 + sub;
        }
      row16_best(bs, bi, qsa_better);
#pragma unroll
      for (int t = 0; t < T; ++t)
        if (doc0 + t * 16 + sub == bi) sc[t] = -INFINITY;
      if (live && sub == 0) {
        const bool some = bs > -INFINITY;
        cand_scores[at + r] = some ? bs : -2.0f;
        cand_ids[at + r] = some ? bi : -1;
      }
    }
  }
}

// sums of 32 products, added up in f64: one f32 chain over the row would double
// the rounding of a score
template <int T, int QT>
__device__ __forceinline__ void qsa_topk_step(const float (&dc)[T][8],
                                              const float (&qc)[QT][8],
                                              double (&total)[T][QT][4]) {
  f32x4_t acc[T][QT];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int u = 0; u < QT; ++u) acc[t][u] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int u = 0; u < QT; ++u)
        acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(
            dc[t][e], qc[u][e], acc[t][u], 0, 0, 0);
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int u = 0; u < QT; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) total[t][u][r] += (double)acc[t][u][r];
}

// numbers k..k+7 of a row; what lies beyond D is zero
__device__ __forceinline__ void qsa_row8(const float* __restrict__ row, int k,
                                         int D, float* v) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = row[k + e < D ? k + e : 0];
    v[e] = k + e < D ? x : 0.f;
  }
}

// waits until at most N loads of the wave are on their way
template <int N>
__device__ __forceinline__ void qsa_topk_wait() {
  static_assert(N < 64, "the counter's range");
  __builtin_amdgcn_s_waitcnt((N & 15) | N >> 4 << 14 | 7 << 4 | 15 << 8);
  asm volatile("" ::: "memory");
}

// Rows of whole 16-byte pieces (D % 4 == 0, aligned).  32 numbers of every row,
// queries and documents, go straight to the wave's LDS, 8 rows of 128 bytes per
// load: read into registers in the matrix cores' layout, the lanes of one load
// touch 16 rows, which the address unit takes four times as long for.  The next
// 32 are on their way while these multiply; no wave waits for another.
// FAR: the index is larger than the last-level cache of 256 MB, where it only drives
// itself out before the next search: loads that do not stay there (100,000 documents, 8
// queries 111.5 -> 97.6 us, 6.3 TB/s; 30,000, which stay, 35.4 -> 44.4).
template <int T, int QT, bool FAR>     // 16*T documents, 16*QT queries
__global__ void __launch_bounds__(256, T + QT <= 2 ? 4 : T + QT <= 3 ? 3 : 1)
qsa_topk_scan(const float* __restrict__ queries,  // [Q, D] L2-normalized
              const float* __restrict__ docs,     // [N, D] L2-normalized
              float* __restrict__ cand_scores,    // [Q, nblk, k]
              int* __restrict__ cand_ids,         // [Q, nblk, k]
              int Qn, int N, int D, int k) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int ROWS = 16 * (T + QT), LOADS = ROWS / 8, STAGE = ROWS * 32;
  constexpr int RING = 4 * 2 * STAGE, PART = 4 * 16 * T * 17;
  __shared__ __attribute__((aligned(16))) float lds[RING > PART ? RING : PART];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  const int doc0 = blockIdx.x * 16 * T, q0 = blockIdx.y * 16 * QT;

  // Rows beyond the end shadow the last one; nothing of theirs is kept.  A
  // row's eight 16-byte pieces are exchanged by its number, which spreads the
  // reads below over the banks.
  const float* row[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = i * 8 + (lane >> 3);
    row[i] = (i < 2 * T
                  ? docs + (long long)min(doc0 + r, N - 1) * D
                  : queries + (long long)min(q0 + r - 16 * T, Qn - 1) * D) +
             ((lane & 7) ^ (r >> 1 & 7)) * 4;
  }

  double total[T][QT][4];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int u = 0; u < QT; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) total[t][u][r] = 0.0;

  const int steps = D / 32;            // whole ones
  float* ring = lds + wave * 2 * STAGE;
  auto fetch = [&](int s, int at) {
    auto to = [&](int i) {
      return (__attribute__((address_space(3))) void*)(ring + at * STAGE + i * 256);
    };
    auto of = [&](int i) {
      return (const __attribute__((address_space(1))) void*)(row[i] + s * 32);
    };
#pragma unroll
    for (int i = 0; i < 2 * T; ++i)
      __builtin_amdgcn_global_load_lds(of(i), to(i), 16, 0, FAR ? QSA_NT : 0);
#pragma unroll
    for (int i = 2 * T; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds(of(i), to(i), 16, 0, 0);
  };
  float dc[T][8], qc[QT][8];
  int at = 0;
  if (wave < steps) fetch(wave, 0);
  for (int s = wave; s < steps; s += 4, at ^= 1) {
    if (s + 4 < steps) {
      fetch(s + 4, at ^ 1);
      qsa_topk_wait<LOADS>();
    } else {
      qsa_topk_wait<0>();
    }
    const float* tile = ring + at * STAGE + col * 32;
    auto take = [&](int i, float* v) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(
            tile + i * 512 + ((hi * 2 + h) ^ (col >> 1)) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[h * 4 + e] = x[e];
      }
    };
#pragma unroll
    for (int t = 0; t < T; ++t) take(t, dc[t]);
#pragma unroll
    for (int u = 0; u < QT; ++u) take(T + u, qc[u]);
    qsa_topk_step<T, QT>(dc, qc, total);
    // the reads are done before the stage is written again
    __builtin_amdgcn_s_waitcnt(0xc07f);            // lgkmcnt(0)
    asm volatile("" ::: "memory");
  }
  if (steps * 32 < D && (steps & 3) == wave) {     // the last, part of a step
    const int kk = steps * 32 + hi * 8;
#pragma unroll
    for (int t = 0; t < T; ++t)
      qsa_row8(docs + (long long)min(doc0 + t * 16 + col, N - 1) * D, kk, D,
               dc[t]);
#pragma unroll
    for (int u = 0; u < QT; ++u)
      qsa_row8(queries + (long long)min(q0 + u * 16 + col, Qn - 1) * D, kk, D,
               qc[u]);
    qsa_topk_step<T, QT>(dc, qc, total);
  }
  __syncthreads();                     // every wave has read its last stage
  qsa_topk_candidates<T, QT>(reinterpret_cast<float (*)[16 * T][17]>(lds),
                             total, doc0, q0, cand_scores, cand_ids, Qn, N, k);
#endif
}

// The same for any other D and alignment, number by number.
template <int T, int QT>
__global__ void __launch_bounds__(256, 2)
qsa_topk_scan_any(const float* __restrict__ queries,
                  const float* __restrict__ docs,
                  float* __restrict__ cand_scores, int* __restrict__ cand_ids,
                  int Qn, int N, int D, int k) {
  __shared__ float part[4][16 * T][17];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  const int doc0 = blockIdx.x * 16 * T, q0 = blockIdx.y * 16 * QT;

  const float* qrow[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u)
    qrow[u] = queries + (long long)min(q0 + u * 16 + col, Qn - 1) * D;
  const float* drow[T];
#pragma unroll
  for (int t = 0; t < T; ++t)
    drow[t] = docs + (long long)min(doc0 + t * 16 + col, N - 1) * D;

  double total[T][QT][4];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int u = 0; u < QT; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) total[t][u][r] = 0.0;

  const int steps = (D + 31) / 32;     // 32 floats of every row, 8 per lane
  float qn[QT][8], dn[T][8];
  auto fetch = [&](int s) {
#pragma unroll
    for (int u = 0; u < QT; ++u) qsa_row8(qrow[u], s * 32 + hi * 8, D, qn[u]);
#pragma unroll
    for (int t = 0; t < T; ++t) qsa_row8(drow[t], s * 32 + hi * 8, D, dn[t]);
  };
  if (wave < steps) fetch(wave);
  for (int s = wave; s < steps; s += 4) {
    float qc[QT][8], dc[T][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int u = 0; u < QT; ++u) qc[u][e] = qn[u][e];
#pragma unroll
      for (int t = 0; t < T; ++t) dc[t][e] = dn[t][e];
    }
    if (s + 4 < steps) fetch(s + 4);
    qsa_topk_step<T, QT>(dc, qc, total);
  }
  qsa_topk_candidates<T, QT>(part, total, doc0, q0, cand_scores, cand_ids, Qn,
                             N, k);
}

// A block per query and group of lists: k rounds, each the best candidate behind
// the last one.  Lists are sorted, so a thread keeps the heads of HEADS of them
// and a round compares heads only.  A block has room for 4096 heads; what more
// lists there are (indexes beyond 262,144 documents, 196,608 or 131,072 with 17
// and more queries) form groups, whose results are merged in turn.  Going through the
// lists beyond 4096 in every round instead cost 2.6 of 4.1 ms for a million
// documents, 16 queries and k = 16.
#define QSA_MERGE_THREADS 512
#define QSA_MERGE_HEADS 8

__global__ void __launch_bounds__(QSA_MERGE_THREADS)
qsa_topk_merge(const float* __restrict__ cand_scores,  // [Q, all, k]
               const int* __restrict__ cand_ids,
               float* __restrict__ out_scores,         // [Q, groups, k]
               int* __restrict__ out_ids, int all, int k) {
  constexpr int NT = QSA_MERGE_THREADS, NH = QSA_MERGE_HEADS, NW = NT / 64;
  const int first = blockIdx.y * NT * NH, lists = min(all - first, NT * NH);
  __shared__ float ws[NW];
  __shared__ int wi[NW];
  const int tid = threadIdx.x, wave = tid >> 6;
  const long long from = ((long long)blockIdx.x * all + first) * k;
  const float* cs = cand_scores + from;
  const int* ci = cand_ids + from;
  float hs[NH];
  int hd[NH], at[NH];                  // id -1: the list is used up
#pragma unroll
  for (int j = 0; j < NH; ++j) {
    at[j] = (tid + j * NT) * k;
    const bool in = tid + j * NT < lists;
    hd[j] = in ? ci[at[j]] : -1;
    hs[j] = in ? cs[at[j]] : 0.f;
  }
  float last_s = INFINITY;
  int last_i = -1;
  for (int r = 0; r < k; ++r) {
    float bs = -INFINITY;
    int bi = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < NH; ++j)
      if (hd[j] >= 0 && qsa_better(hs[j], hd[j], bs, bi)) {
        bs = hs[j];
        bi = hd[j];
      }
    wave_best(bs, bi, qsa_better);
    __syncthreads();                   // the round before has been read
    if ((tid & 63) == 0) {
      ws[wave] = bs;
      wi[wave] = bi;
    }
    __syncthreads();
    last_s = ws[0];
    last_i = wi[0];
#pragma unroll
    for (int w = 1; w < NW; ++w)
      if (qsa_better(ws[w], wi[w], last_s, last_i)) {
        last_s = ws[w];
        last_i = wi[w];
      }
    const bool some = last_s > -INFINITY;
    if (tid == 0) {
      const long long to =
          ((long long)blockIdx.x * gridDim.y + blockIdx.y) * k + r;
      out_scores[to] = some ? last_s : -2.0f;
      out_ids[to] = some ? last_i : -1;
    }
#pragma unroll
    for (int j = 0; j < NH; ++j)
      if (hd[j] >= 0 && hd[j] == last_i) {        // its owner moves on
        ++at[j];
        const bool in = at[j] < (tid + j * NT + 1) * k;
        hd[j] = in ? ci[at[j]] : -1;
        hs[j] = in ? cs[at[j]] : 0.f;
      }
  }
}

// Queries from the host's pinned memory, a read of some 10 to 100 KB over the bus
// that the scan's blocks would each repeat.
__global__ void __launch_bounds__(256)
qsa_topk_fetch(const float* __restrict__ host, float* __restrict__ queries,
               long long n) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i + 4 <= n) {
    *reinterpret_cast<float4*>(queries + i) =
        *reinterpret_cast<const float4*>(host + i);
  } else {
    for (long long j = i; j < n; ++j) queries[j] = host[j];
  }
}

extern "C" void qsa_topk_fetch_launch(const float* host, float* queries,
                                      long long n, hipStream_t stream) {
  hipLaunchKernelGGL(qsa_topk_fetch, dim3((unsigned)((n + 1023) / 1024)),
                     dim3(256), 0, stream, host, queries, n);
}

// A block: 16 documents times the first digit, 16 queries times the second.  Up
// to 16 queries: 16 documents for small indexes, 64 as soon as that gives every
// CU two blocks.  More share a read of the index, 32 queries beside 48 documents
// or 48 beside 32, once that fills the CUs (us at 1536, blocks of 16 documents
// and queries / these: 24 queries of 6000 documents 15.7 / 19.3, 10,000 22.4 /
// 20.6, 100,000 248 / 136; 64 of 3000 14.7 / 20.1, 6000 25.5 / 21.0).  33 to 48
// queries are one read where 32 at a time take two (100,000: 195 and 269).
static int qsa_topk_tile(long long Q, long long N) {
  if (Q <= 16) return N < 64 * 512 ? 11 : 41;
  if ((Q + 31) / 32 * N < 8192) return 11;
  return Q > 32 && Q <= 48 ? 23 : 32;
}

// Documents per block.
extern "C" int qsa_topk_block_docs(long long Q, long long N) {
  return qsa_topk_tile(Q, N) / 10 * 16;
}

extern "C" void qsa_topk_scan_launch(const float* queries, const float* docs,
                                     float* cand_scores, int* cand_ids, int Q,
                                     int N, int D, int k, int nblk,
                                     hipStream_t stream) {
  if (N == 0) return;
  const bool vec = D % 4 == 0 && ((reinterpret_cast<uintptr_t>(queries) |
                                   reinterpret_cast<uintptr_t>(docs)) &
                                  15) == 0;
#define QSA_SCAN(T, QT)                                                      \
  {                                                                          \
    const dim3 grid(nblk, (Q + 16 * QT - 1) / (16 * QT));                    \
    if (vec && (long long)N * D * 4 > QSA_LLC)                               \
      hipLaunchKernelGGL((qsa_topk_scan<T, QT, true>), grid, dim3(256), 0,   \
                         stream, queries, docs, cand_scores, cand_ids, Q, N, \
                         D, k);                                              \
    else if (vec)                                                            \
      hipLaunchKernelGGL((qsa_topk_scan<T, QT, false>), grid, dim3(256), 0,  \
                         stream, queries, docs, cand_scores, cand_ids, Q, N, \
                         D, k);                                              \
    else                                                                     \
      hipLaunchKernelGGL((qsa_topk_scan_any<T, QT>), grid, dim3(256), 0,     \
                         stream, queries, docs, cand_scores, cand_ids, Q, N, \
                         D, k);                                              \
  }
  switch (qsa_topk_tile(Q, N)) {
    case 11: QSA_SCAN(1, 1) break;
    case 41: QSA_SCAN(4, 1) break;
    case 32: QSA_SCAN(3, 2) break;
    default: QSA_SCAN(2, 3)
  }
#undef QSA_SCAN
}

// Lists that a merge leaves of `lists`: one is the result.
extern "C" int qsa_topk_groups(int lists) {
  const int n = QSA_MERGE_THREADS * QSA_MERGE_HEADS;
  return lists > n ? (int)(((long long)lists + n - 1) / n) : 1;
}

extern "C" void qsa_topk_merge_launch(const float* cand_scores,
                                      const int* cand_ids, float* out_scores,
                                      int* out_ids, int Q, int lists, int k,
                                      hipStream_t stream) {
  const dim3 grid(Q, qsa_topk_groups(lists));
  hipLaunchKernelGGL(qsa_topk_merge, grid, dim3(QSA_MERGE_THREADS), 0, stream,
                     cand_scores, cand_ids, out_scores, out_ids, lists, k);
}
