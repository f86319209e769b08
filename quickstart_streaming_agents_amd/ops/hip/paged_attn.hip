// Paged-attention DECODE for CDNA4 (gfx950) — the K4 hot op, on MFMA.
//
// Replaces the reference's managed-LLM call (ML_PREDICT 'llm_textgen_model',
// terraform/core/main.tf:461) with on-GPU batched decode attention over a
// paged KV cache resident in 288 GB HBM3E.
//
// Design (flash decoding; a block of NW waves per (row b, kv head, share of the
// pages), a wave per page in turn):
//   - All R GQA query heads of a kv head compute TOGETHER on the matrix
//     cores: scores via mfma_f32_16x16x32_bf16 with A = K-tile
//     [16 pos x 32 k] and B = Q [32 k x 16 heads] (heads pad to 16), PV
//     via A = P [16 heads x 32 pos] (packed bf16, redistributed by lane
//     swaps) and B = V^T [32 pos x 16 dims].  Every KV byte is
//     read exactly once.
//   - K cache layout [page, kvh, D/8, 64, 8] (d-major x8): a page's fragments
//     are loads of four 256-byte pieces, and the next page's are under way while
//     one is multiplied.  V cache layout [page, kvh, D, 64] (transposed, pos
//     minor): its fragments would be pieces of 16 bytes, four times the address
//     cycles, so a page goes into the wave's LDS in whole lines and is read from
//     there (8 rows of 500-900 keys 16.7 -> 14.6 us).
//   - The waves of a block merge in LDS.  One block per (row, kv head) stores
//     the result; several leave (o, m, l) for qsa_attn_reduce.
//   - FUSE is a decoding step's attention: q is rotated in registers, and the
//     wave with the last page writes the rotated new key and the new value to
//     the cache, so that no launch has to come before.  It puts both in their
//     place among what it has read: waiting for its own stores cost a round
//     trip to memory.
// 192 rows of 400-1000 keys, 32/8 heads of 128: 131 -> 124 us, of which 105 are
// the reads (5.2 TB/s of keys and values, 5.5 with the rest of last pages) and the
// rest the 128 lines per row and head that a transposed value touches, whatever the
// width of the stores or their cache policy (64-byte pieces, whole lines and
// write-through were the same).
//
// The online softmax runs per head-column in registers: column max/sum
// reduce by two lane swaps (the 4 hi-lane groups of a column).
#include <algorithm>
#include <type_traits>

#include "lm_common.h"

#define QSA_PAGE 64

using bf16x8_a = __attribute__((ext_vector_type(8))) short;
using f32x4_a = __attribute__((ext_vector_type(4))) float;

// place of element k of a step's row in packed activations (skinny_stream.h)
__device__ __forceinline__ long long qsa_step_at(int row, int k, int mt) {
  return ((long long)(k >> 5) * mt + (row >> 4)) * 512 +
         ((row & 15) + ((k >> 3) & 3) * 16) * 8 + (k & 7);
}

struct DecodeArgs {
  const unsigned short* q;             // [B, QH, D], row stride qstride
  const unsigned short* kc;            // [P, KVH, D/8, 64, 8]
  const unsigned short* vc;            // [P, KVH, D, 64]
  const int* block_table;              // [B, max_pages]
  const int* seq_lens;                 // [B]
  float* part_o;                       // [B, QH, NS, D]
  float* part_ml;                      // [B, QH, NS, 2]
  unsigned short* out;                 // NS == 1: [B, QH, D], or packed rows
  // FUSE
  const unsigned short* k;             // [B, KVH, D], row stride kvstride
  const unsigned short* v;
  unsigned short* kw;                  // the caches again, to write
  unsigned short* vw;
  const float* cos_t;                  // [positions, D/2]
  const float* sin_t;
  float scale;
  int QH, KVH, max_pages, NS, mt;      // mt: row tiles of packed rows, or 0
  long long qstride, kvstride;
  // blocks beyond the attention's read these (in 16 bytes)
  int blocks;
  const u32x4_v* warm[2];
  long long warm_n[2];
  // keys of all `rows` beyond which pages are read past the last-level cache
  int rows;
  float far_keys;
};

// Reads memory for the launches that follow, towards the last-level cache.
template <int THREADS>
__device__ __forceinline__ void qsa_warm(const u32x4_v* at, long long n,
                                         int block, int blocks) {
  constexpr int U = 8;
  for (long long i = (long long)block * THREADS * U + threadIdx.x; i < n;
       i += (long long)blocks * THREADS * U) {
    u32x4_v v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[u] = at[min(i + u * THREADS, n - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u) asm volatile("" ::"v"(v[u]));
  }
}

// Rotate elements k0.. and k0 + D/2.. of a row held in two fragments.  Which product is
// fused is not left to the compiler, who decides it for each kernel, so that a query has
// the same bits whether it is turned on its way into the attention or before it: the
// cosine's, but SIN in the second half of a prompt's keys.
template <bool SIN = false>
__device__ __forceinline__ void rotate_pair(bf16x8_a& a, bf16x8_a& b,
                                            const float* c, const float* s) {
  u32x4_v u = __builtin_bit_cast(u32x4_v, a), v = __builtin_bit_cast(u32x4_v, b);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float2 x = bf16x2_to_f32x2(u[e]), y = bf16x2_to_f32x2(v[e]);
    const float c0 = c[2 * e], c1 = c[2 * e + 1];
    const float s0 = s[2 * e], s1 = s[2 * e + 1];
    u[e] = cvt_bf16x2(fmaf(x.x, c0, -(y.x * s0)), fmaf(x.y, c1, -(y.y * s1)));
    v[e] = SIN ? cvt_bf16x2(fmaf(x.x, s0, y.x * c0), fmaf(x.y, s1, y.y * c1))
               : cvt_bf16x2(fmaf(y.x, c0, x.x * s0), fmaf(y.y, c1, x.y * s1));
  }
  a = __builtin_bit_cast(bf16x8_a, u);
  b = __builtin_bit_cast(bf16x8_a, v);
}

// Up to 63 of a wave's loads under way, whatever it stored or read from LDS.  It
// counts, so no load may pass it either way (tests/test_isa_audit.py looks at what
// stands before it).
template <int N> __device__ __forceinline__ void wait_vm() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | 7 << 4 | 15 << 8);
  asm volatile("" ::: "memory");
}

// How pages are read: STAY, to be found in the last-level cache by the next step, or
// PAST it (see the launch).  STAY_BUFFER is STAY in a kernel that has both, with keys
// by buffer loads, so that an audit of its counted waits tells the two apart.
enum { STAY, PAST, STAY_BUFFER };

template <int D, int NW, bool FUSE, int PAGES>
__device__ __forceinline__ void qsa_paged_attn(const DecodeArgs& p,
                                               unsigned short* vlds, float* ml) {
  constexpr bool FAR = PAGES == PAST;
  constexpr int KSTEPS = D / 32;      // QK^T k-steps (4 for D=128)
  constexpr int DTILES = D / 16;      // PV d-tiles (8 for D=128)
  constexpr int VT = D * QSA_PAGE;    // elements of a value page
  constexpr int KL = 4 * KSTEPS;      // loads of a wave for a page's keys
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int split = blockIdx.x % p.NS;
  const int bk = blockIdx.x / p.NS;
  const int b = bk / p.KVH;
  const int kvh = bk % p.KVH;
  const int R = p.QH / p.KVH;
  const int first = split * NW + wave, step = NW * p.NS;
  // scalar loads: as a vector load a page's number, newer than the loads under
  // way, would have waited for all of them
  const auto btab = (const __attribute__((address_space(4))) int*)(
      p.block_table + (long long)b * p.max_pages);
  // side by side: the first pages' numbers wait for no length
  int page = btab[min(first, p.max_pages - 1)];
  int next = btab[min(first + step, p.max_pages - 1)];
  const int seqlen = p.seq_lens[b];
  const int npages = (seqlen + QSA_PAGE - 1) / QSA_PAGE;
  const int col = lane & 15;          // head col (scores) / dim col (PV)
  const int hi = lane >> 4;           // 4 hi-lane groups

  float m = -3.0e38f, lsum = 0.f;
  f32x4_a o_acc[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt)
    o_acc[dt] = (f32x4_a){0.f, 0.f, 0.f, 0.f};

  if (first < npages) {               // uniform over the wave
    // ---- Q B-fragments: lane holds Q[head=col][k = ks*32 + hi*8 + e] ----
    const int qh_l = kvh * R + min(col, R - 1);   // clamp: pad heads compute
    const unsigned short* qrow =
        p.q + (long long)b * p.qstride + (long long)qh_l * D;
    bf16x8_a qf[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks)
      qf[ks] = *reinterpret_cast<const bf16x8_a*>(qrow + ks * 32 + hi * 8);
    auto load_k = [&](int page, bf16x8_a (&kf)[4][KSTEPS]) {
      const unsigned short* kbase =
          p.kc + ((((long long)page * p.KVH + kvh) * (D / 8)) * QSA_PAGE) * 8;
      if constexpr (PAGES == STAY_BUFFER) {
        const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
            (void*)kbase, 0, VT * 2, 0x00027000);
#pragma unroll
        for (int pt = 0; pt < 4; ++pt)
#pragma unroll
          for (int ks = 0; ks < KSTEPS; ++ks)
            kf[pt][ks] = __builtin_bit_cast(
                bf16x8_a, __builtin_amdgcn_raw_buffer_load_b128(
                              rk, hi * 1024 + col * 16 + pt * 256, ks * 4096, 0));
        return;
      }
#pragma unroll
      for (int pt = 0; pt < 4; ++pt)
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          const bf16x8_a* at = reinterpret_cast<const bf16x8_a*>(
              kbase + ((ks * 4 + hi) * QSA_PAGE + pt * 16 + col) * 8);
          kf[pt][ks] = FAR ? __builtin_nontemporal_load(at) : *at;
        }
    };
    // Values go straight to the wave's LDS, 8 rows of 128 bytes at a time, a
    // row's segments exchanged by its number (the reads below then spread over
    // the banks).  By buffer loads: behind a global one to LDS the compiler waits
    // for everything that is under way wherever it has to wait for anything.
    unsigned short* vl = vlds + wave * VT;
    const unsigned int voff =
        ((lane >> 3) * QSA_PAGE + ((lane & 7) ^ (lane >> 3)) * 8) * 2;
    auto load_v = [&](int page) {
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(p.vc + ((long long)page * p.KVH + kvh) * VT), 0, VT * 2,
          0x00027000);
#pragma unroll
      for (int i = 0; i < D / 8; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rv, (__attribute__((address_space(3))) void*)(vl + i * 512), 16,
            voff, i * 1024, 0, FAR ? QSA_NT : 0);
    };
    bf16x8_a kf[4][KSTEPS];
    load_k(page, kf);
    // the new key, in the same order: every lane's column is a copy; and value
    bf16x8_a kn[FUSE ? KSTEPS : 1];
    unsigned short vn[FUSE ? D / 64 : 1];
    float cs[FUSE ? KSTEPS / 2 : 1][8], sn[FUSE ? KSTEPS / 2 : 1][8];
    if constexpr (FUSE) {
      const long long row = (long long)b * p.kvstride + (long long)kvh * D;
      const unsigned short* krow = p.k + row;
#pragma unroll
      for (int i = 0; i < D / 64; ++i) vn[i] = p.v[row + i * 64 + lane];
      const long long at = (long long)(seqlen - 1) * (D / 2) + hi * 8;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
        kn[ks] = *reinterpret_cast<const bf16x8_a*>(krow + ks * 32 + hi * 8);
#pragma unroll
      for (int ks = 0; ks < KSTEPS / 2; ++ks) {
        ldv<float, 8>(p.cos_t + at + ks * 32, cs[ks]);
        ldv<float, 8>(p.sin_t + at + ks * 32, sn[ks]);
      }
    }
    load_v(page);                     // behind all that the scores wait for
    if constexpr (FUSE) {
#pragma unroll
      for (int ks = 0; ks < KSTEPS / 2; ++ks) {
        rotate_pair(qf[ks], qf[ks + KSTEPS / 2], cs[ks], sn[ks]);
        rotate_pair(kn[ks], kn[ks + KSTEPS / 2], cs[ks], sn[ks]);
      }
    }

    // Page pi; the keys of the wave's next one are asked for once these have been
    // multiplied, its values once these have (values only behind the page's own
    // keys: 100 rows of 400-1000 keys +1 %, 33 of 3000-4000 -3 %).  The last page is
    // code of its own, or the waits of both would be for all that is under way.
    // patch: the row's last page, where the new token has its place.
    auto walk = [&](int pi, auto last) {
      const int after = btab[min(pi + 2 * step, p.max_pages - 1)];
      const int nvalid = min(seqlen - pi * QSA_PAGE, QSA_PAGE);
      const int pin = nvalid - 1;
      const bool patch = FUSE && last.value && pi == npages - 1;
      if (patch) {
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
          for (int pt = 0; pt < 4; ++pt)
            if (pt * 16 + col == pin) kf[pt][ks] = kn[ks];
      }
      // ---- scores: 4 pos-tiles x KSTEPS MFMAs ---------------------------
      // A-frag: lane holds K[pos = pt*16 + col][k = ks*32 + hi*8 + e]
      f32x4_a sc[4];
#pragma unroll
      for (int pt = 0; pt < 4; ++pt) {
        f32x4_a acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[pt][ks], qf[ks],
                                                        acc, 0, 0, 0);
        sc[pt] = acc;
      }
      if constexpr (!last.value) load_k(next, kf);
      // scale + mask invalid positions; C layout: row pos = hi*4 + r,
      // col head = lane&15 -> lane's r-th value is position pt*16 + hi*4 + r
      float pagemax = -3.0e38f;
#pragma unroll
      for (int pt = 0; pt < 4; ++pt) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int pos = pt * 16 + hi * 4 + r;
          float v = (pos < nvalid) ? sc[pt][r] * p.scale : -3.0e38f;
          sc[pt][r] = v;
          pagemax = fmaxf(pagemax, v);
        }
      }
      // column (per-head) max across the 4 hi groups
      pagemax = rows_max(pagemax);
      const float m_new = fmaxf(m, pagemax);
      float alpha = __expf(m - m_new);
      if (m <= -3.0e38f) alpha = 0.f;
      m = m_new;
      // o_acc element (dt, r) belongs to OUTPUT ROW hi*4 + r (the PV
      // C-layout), while alpha lives per score COLUMN (this lane's l&15):
      // fetch each row's own alpha from the lane holding that column
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float alpha_r = __shfl(alpha, hi * 4 + r, 16);
#pragma unroll
        for (int dt = 0; dt < DTILES; ++dt) o_acc[dt][r] *= alpha_r;
      }
      // P = exp(sc - m) (invalid -> 0), packed bf16x2 per tile quad
      unsigned int ppk[8];   // tile pt -> 2 uints (4 bf16 = quads r0..3)
      float psum = 0.f;
#pragma unroll
      for (int pt = 0; pt < 4; ++pt) {
        float pr[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          pr[r] = sc[pt][r] > -1.0e38f ? __expf(sc[pt][r] - m_new) : 0.f;
          psum += pr[r];
        }
        ppk[pt * 2] = cvt_bf16x2(pr[0], pr[1]);
        ppk[pt * 2 + 1] = cvt_bf16x2(pr[2], pr[3]);
      }
      psum = rows_sum(psum);
      lsum = lsum * alpha + psum;

      // the values are there; the next page's keys, behind them, need not be
      wait_vm<last.value ? 0 : KL>();
      if (patch) {
#pragma unroll
        for (int i = 0; i < D; i += 64) {
          const int d = i + lane;
          vl[d * 64 + ((pin >> 3) ^ (d & 7)) * 8 + (pin & 7)] = vn[i / 64];
          p.vw[((long long)page * p.KVH + kvh) * VT + d * 64 + pin] = vn[i / 64];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
      }
      // ---- PV: two 32-pos halves ---------------------------------------
      // A-frag needs lane (head=col, hi) to hold P[head][pos = hi*8 + e]: packed
      // pairs of the groups 2hi & 3 and the next of tile half*2 + (hi>>1).  Of
      // two tiles' groups (0 1 2 3) and (4 5 6 7) a swap of halves makes (0 1 4
      // 5) and (2 3 6 7), and one of rows (0 2 4 6) and (1 3 5 7), which is that
      // (16 exchanges through LDS: a step of one row 524 us, 521 so; of 24 rows of
      // 800-2000 keys 937 and 931).
      // B-frag: lane holds V^T[pos = half*32 + hi*8 + e][d = dt*16+col]
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u32x4_v pu;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const auto x = __builtin_amdgcn_permlane32_swap(
              ppk[half * 4 + w], ppk[half * 4 + 2 + w], false, false);
          const auto y =
              __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
          pu[w] = y[0];
          pu[2 + w] = y[1];
        }
        const bf16x8_a pa = __builtin_bit_cast(bf16x8_a, pu);
        const unsigned short* vr =
            vl + col * 64 + ((half * 4 + hi) ^ (col & 7)) * 8;
        bf16x8_a vf[DTILES];
#pragma unroll
        for (int dt = 0; dt < DTILES; ++dt)
          vf[dt] = *reinterpret_cast<const bf16x8_a*>(vr + dt * 1024);
#pragma unroll
        for (int dt = 0; dt < DTILES; ++dt)
          o_acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              pa, vf[dt], o_acc[dt], 0, 0, 0);
      }
      if (patch) {                     // the key's lines: 8 positions each
#pragma unroll
        for (int pt = 0; pt < 4; ++pt)
          if (pt * 16 + col == pin) {
            unsigned short* kw =
                p.kw + ((long long)page * p.KVH + kvh) * VT;
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks)
              *reinterpret_cast<bf16x8_a*>(
                  kw + ((ks * 4 + hi) * QSA_PAGE + pt * 16 + col) * 8) =
                  kf[pt][ks];
          }
      }
      if constexpr (!last.value) {
        // all of the values have been read when the next page's come
        __builtin_amdgcn_s_waitcnt(0xc07f);       // lgkmcnt(0)
        asm volatile("" ::: "memory");
        load_v(next);
        asm volatile("" ::: "memory");            // and no key's load before
        page = next;
        next = after;
      }
    };
    int pi = first;
    for (; pi + step < npages; pi += step) walk(pi, std::false_type{});
    walk(pi, std::true_type{});
  }

  // ---- the waves of the block meet: O C-layout row = head = hi*4 + r -----
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  float* os = reinterpret_cast<float*>(vlds);     // [NW][VT / 2]
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int head = hi * 4 + r;
    if (head < R)
#pragma unroll
      for (int dt = 0; dt < DTILES; ++dt)
        os[wave * (VT / 2) + head * D + dt * 16 + col] = o_acc[dt][r];
  }
  if (lane < 16) {
    ml[wave * 16 + lane] = m;
    ml[NW * 16 + wave * 16 + lane] = lsum;
  }
  __syncthreads();
  for (int i = tid; i < R * D; i += NW * 64) {
    const int head = i / D, d = i % D;
    float M = -3.0e38f;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, ml[w * 16 + head]);
    float L = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float ls = ml[NW * 16 + w * 16 + head];
      // a wave without keys: no weight, whatever M is
      const float f = ls > 0.f ? __expf(ml[w * 16 + head] - M) : 0.f;
      L += f * ls;
      acc += f * os[w * (VT / 2) + i];
    }
    const int qh = kvh * R + head;
    if (p.NS == 1) {
      const unsigned short v = cvt_bf16(L > 0.f ? acc / L : 0.f);
      if (p.mt)
        p.out[qsa_step_at(b, qh * D + d, p.mt)] = v;
      else
        p.out[((long long)b * p.QH + qh) * D + d] = v;
    } else {
      const long long at = ((long long)b * p.QH + qh) * p.NS + split;
      p.part_o[at * D + d] = acc;
      if (d == 0)
        *reinterpret_cast<float2*>(p.part_ml + at * 2) = make_float2(M, L);
    }
  }
}

// the blocks beyond the attention's
template <int NW>
__device__ __forceinline__ bool qsa_warmed(const DecodeArgs& p) {
  if ((int)blockIdx.x < p.blocks) return false;
  for (int i = 0; i < 2; ++i)
    qsa_warm<NW * 64>(p.warm[i], p.warm_n[i], blockIdx.x - p.blocks,
                      gridDim.x - p.blocks);
  return true;
}

// LDS: a wave's values, afterwards its part of the output [R][D], and its maxima and
// sums
#define QSA_DECODE_LDS                                                      \
  __shared__ __attribute__((aligned(16)))                                   \
      unsigned short vlds[NW * D * QSA_PAGE];                               \
  __shared__ float ml[2 * NW * 16];                                         \
  if (FUSE && qsa_warmed<NW>(p)) return

template <int D, int NW, bool FUSE>
__global__ void __launch_bounds__(NW * 64, NW == 4 ? 2 : 1)
qsa_paged_attn_mfma(DecodeArgs p) {
  QSA_DECODE_LDS;
  qsa_paged_attn<D, NW, FUSE, STAY>(p, vlds, ml);
}
// of a table that has room for far more than is live, perhaps
template <int D, int NW, bool FUSE>
__global__ void __launch_bounds__(NW * 64, NW == 4 ? 2 : 1)
qsa_paged_attn_far(DecodeArgs p) {
  QSA_DECODE_LDS;
  if (wave_total(p.seq_lens, p.rows, [](int n) { return (float)max(n, 0); }) >
      p.far_keys)
    qsa_paged_attn<D, NW, FUSE, PAST>(p, vlds, ml);
  else
    qsa_paged_attn<D, NW, FUSE, STAY_BUFFER>(p, vlds, ml);
}
#undef QSA_DECODE_LDS

template <int D>
__global__ void __launch_bounds__(128)
qsa_attn_reduce(const float* __restrict__ part_o,   // [rows, NS, D]
                const float* __restrict__ part_ml,  // [rows, NS, 2]
                unsigned short* __restrict__ out,   // [rows, D], or packed
                int NS, int QH, int mt) {
  const long long row = blockIdx.x;
  const int d = threadIdx.x;  // D threads
  const float* ml = part_ml + row * NS * 2;
  const float* po = part_o + row * NS * D + d;
  // The first shares whole, statistics and results, before any is waited for: the
  // results used to be asked for once the largest was known (16 rows of 1536-2048
  // keys, 16 layers: 674.8 us a step, 670.3 now; 2 rows 506 and 500).
  constexpr int U = 4;
  float m0[U], l0[U], o0[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int s = min(u, NS - 1);                   // beyond the last: again
    o0[u] = po[s * D];
    m0[u] = ml[2 * s];
    l0[u] = ml[2 * s + 1];
  }
  __builtin_amdgcn_sched_barrier(0);
  float M = -3.0e38f;
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (u < NS && l0[u] > 0.f) M = fmaxf(M, m0[u]);
#pragma unroll 4
  for (int s = U; s < NS; ++s)
    if (ml[2 * s + 1] > 0.f) M = fmaxf(M, ml[2 * s]);
  float L = 0.f, acc = 0.f;
  auto add = [&](float m, float l, float o) {
    const float w = l > 0.f ? __expf(m - M) : 0.f;
    L += w * l;
    acc += w * o;
  };
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (u < NS) add(m0[u], l0[u], o0[u]);
#pragma unroll 4
  for (int s = U; s < NS; ++s) add(ml[2 * s], ml[2 * s + 1], po[s * D]);
  const unsigned short v = cvt_bf16((L > 0.f) ? acc / L : 0.f);
  if (mt)
    out[qsa_step_at((int)(row / QH), (int)(row % QH) * D + d, mt)] = v;
  else
    out[row * D + d] = v;
}

// Waves of a block and blocks per (row, kv head), of which several cost a second
// launch (3 to 4 us).  Up to 16 pages a block of eight waves is over before one
// of several and the merge (32/8 heads of 128, 1 row of 700 keys 11.5 us against
// 13.1, 16 rows 16.5 / 19.1); four once they share CUs (48 rows 38.1 / 41.6).
// Longer rows: from 129 pairs eight waves alone (24 rows of 1000-2000 keys 35.8
// us, three blocks of four 43; 28 of 2500-4000 77 / 84), from 257 four alone (48 of
// 1000-2000 69.8, two blocks 70.4; 63: 84.4 / 89.4), but three of four while the
// chip's second round is nearly empty and rows are long (33 of 3000-4096 102 / 111);
// below, what fills the chip (8 of 1000-2000 19.1, eight blocks of four 21.5; 12
// 23.0 / 27.9).
// max_pages is the table's width, since the rows' lengths are on the device: in
// a table for longer rows, as a captured step's is, short ones of up to 128 pairs
// are split, with the merge and without the read-ahead below.  us, a table as wide
// as the longest row / of 33 / 128 / 256 pages: 1 row of 700 keys 8.6 / 9.2 / 11.1 /
// 13.8; 4 of 500-900 11.6 / 10.8 / 14.2 / 14.5; 8 11.8 / 14.4 / 14.2 / 14.3; 16
// 17.1 / 17.8 / 17.5 / 17.5; of 60-100 keys 1 row 6.5 / 8.7 / 10.1 / 12.9, 16 6.8 /
// 9.7 / 9.6 / 9.7; from 24 rows on and beyond 1000 keys the width is nothing.  Rows
// of 12,000 to 16,000 keys follow the same rule: 8 93 us, 24 252, 64 652 (5.6 TB/s).
extern "C" void qsa_paged_attn_split(int B, int QH, int KVH, int max_pages,
                                     int D, int* waves, int* splits) {
  const long long heads = (long long)B * KVH;
  const bool few = max_pages <= 16;
  *waves = heads > 256 || max_pages <= 4 || (heads <= 48 && !few) ? 4 : 8;
  *splits = 1;
  if (heads == 0) return;
  if (heads > 256) {
    if (heads < 384 && max_pages > 32) *splits = 3;
  } else if (!few && heads <= 128) {
    const long long fill = (2048 + 4 * heads - 1) / (4 * heads);
    *splits = heads > 64   ? 2
              : heads > 48 ? 4
                           : (int)std::min<long long>(fill, (max_pages + 7) / 8);
  }
}

extern "C" void qsa_paged_attn_mfma_launch(
    const unsigned short* q, const unsigned short* k, const unsigned short* v,
    unsigned short* kc, unsigned short* vc, const float* cos_t,
    const float* sin_t, const int* block_table, const int* seq_lens,
    float* part_o, float* part_ml, unsigned short* out, float scale, int B,
    int QH, int KVH, int max_pages, int D, long long qstride,
    long long kvstride, int waves, int NS, int mt, const void* const* warm,
    const long long* warm_bytes, hipStream_t stream) {
  DecodeArgs p{q, kc, vc, block_table, seq_lens, part_o, part_ml, out,
               k, v, kc, vc, cos_t, sin_t, scale, QH, KVH, max_pages,
               NS, mt, qstride, kvstride, 0, {nullptr, nullptr}, {0, 0},
               B, (float)(QSA_FAR_PAGES / (KVH * D * 4))};
  dim3 grid((unsigned)((long long)B * KVH * NS)), block(waves * 64);
  if (grid.x == 0) return;
  p.blocks = (int)grid.x;
  // Few blocks of few pages leave most of the chip idle for some 9 us: as much
  // as memory delivers meanwhile, or nothing, since a projection whose weights
  // are there in part waits for the rest.  2048-wide decoder, 16 layers, output
  // and down projections of 21 MB: 8 rows 518 -> 500 us a step; cut to 24 MB of a
  // 4096-wide one's 75 it cost 1-2%.  Up to 4 rows those projections are as fast on
  // weights from memory, and the attention is over sooner without the other blocks: 1
  // row of 700 keys 461 us without, 468 with, of 120 425 and 445; 3 and 4 rows level.
  const long long bytes = warm_bytes[0] + warm_bytes[1];
  if (k && NS == 1 && B > 4 && grid.x <= 64 && bytes >= 16 &&
      bytes <= 24 << 20) {
    for (int i = 0; i < 2; ++i) {
      p.warm[i] = static_cast<const u32x4_v*>(warm[i]);
      p.warm_n[i] = warm_bytes[i] / 16;
    }
    grid.x = 256;
  }
  // A step reads the pages of all layers and all weights, once.  Pages of small
  // batches may stay in the last-level cache for the next step (the weights are read
  // past it, skinny_stream.h); large ones would drive each other out.  us a step, with
  // loads that stay / that do not: 2048-wide, 8 layers, 4 rows of 600-1000 keys (13 MB a
  // layer) 321 / 350; 16 layers of 64-dim heads, 8 rows of 300-600 (8 MB) 585 / 609, 24
  // of 800-2000 (80 MB) 987 / 971; 4096-wide, 8 layers, 1 row of 900 (4 MB) 504 / 522,
  // 16 of 1536-2048 (134 MB) 722 / 702, 192 of 400-1000 (600 MB) 2295 / 2180.
  // What counts are the keys that are there, which only the device knows: a captured
  // step's table has room for `max_batch` rows of `max_seq_len`, so where that exceeds
  // the line the kernel sums them up (us a step by room / by keys: 4096-wide, 4 rows of
  // 600-1000 in a table of 256 pages 528 / 515, 4 live ones of 32 656 / 633; 1 row of
  // 700 in 512 pages of the 16 layers 690 / 676; the sum itself: 192 rows 2111 / 2115).
  const bool far =
      (long long)B * max_pages * KVH * D * QSA_PAGE * 4 > QSA_FAR_PAGES;
#define QSA_DECODE(DD, NW)                                                  \
  if (D == DD && waves == NW) {                                             \
    if (k && far) QSA_DECODE_AS(qsa_paged_attn_far, DD, NW, true);          \
    else if (k) QSA_DECODE_AS(qsa_paged_attn_mfma, DD, NW, true);           \
    else if (far) QSA_DECODE_AS(qsa_paged_attn_far, DD, NW, false);         \
    else QSA_DECODE_AS(qsa_paged_attn_mfma, DD, NW, false);                 \
  }
#define QSA_DECODE_AS(NAME, DD, NW, FUSE)                                   \
  hipLaunchKernelGGL((NAME<DD, NW, FUSE>), grid, block, 0, stream, p)
  QSA_DECODE(128, 4) QSA_DECODE(128, 8) QSA_DECODE(64, 4) QSA_DECODE(64, 8)
#undef QSA_DECODE
#undef QSA_DECODE_AS
  if (NS == 1) return;
  if (D == 128)
    hipLaunchKernelGGL((qsa_attn_reduce<128>), dim3(B * QH), dim3(128), 0,
                       stream, part_o, part_ml, out, NS, QH, mt);
  else
    hipLaunchKernelGGL((qsa_attn_reduce<64>), dim3(B * QH), dim3(64), 0,
                       stream, part_o, part_ml, out, NS, QH, mt);
}

// ---------------------------------------------------------------------------
// KV-cache writers.  K layout [page, kvh, D/8, 64, 8]; V layout
// [page, kvh, D, 64] (transposed for the PV B-fragment stream).
// ---------------------------------------------------------------------------

// Fused decode-step RoPE + KV append: rotates q in place, rotates k and
// writes it (and v) STRAIGHT into the paged cache.
__global__ void
qsa_rope_kv_append(unsigned short* __restrict__ q,        // [B, QH, D]
                   const unsigned short* __restrict__ k,  // [B, KVH, D]
                   const unsigned short* __restrict__ v,  // [B, KVH, D]
                   unsigned short* __restrict__ kc, unsigned short* __restrict__ vc,
                   const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                   const int* __restrict__ block_table,
                   const int* __restrict__ seq_lens,
                   int B, int QH, int KVH, int D, int max_pages,
                   long long qstride, long long kvstride) {
  const int nheads = QH + KVH;
  const int b = blockIdx.x / nheads;
  const int h = blockIdx.x % nheads;
  const int half = D / 2;
  const int d = threadIdx.x;
  const int pos = seq_lens[b] - 1;
  if (pos < 0) return;
  const long long toff = (long long)pos * half + (d % half);
  const float c = cos_t[toff], s = sin_t[toff];
  if (h < QH) {
    if (d >= half) return;
    unsigned short* base = q + (long long)b * qstride + (long long)h * D;
    const float x0 = bf16_to_f32(base[d]);
    const float x1 = bf16_to_f32(base[d + half]);
    base[d] = f32_to_bf16(x0 * c - x1 * s);
    base[d + half] = f32_to_bf16(x0 * s + x1 * c);
    return;
  }
  if (d >= D) return;
  const int kvh = h - QH;
  const int page = block_table[(long long)b * max_pages + pos / QSA_PAGE];
  const int pin = pos % QSA_PAGE;
  const unsigned short* kbase =
      k + (long long)b * kvstride + (long long)kvh * D;
  const int dl = d % half;
  const float x0 = bf16_to_f32(kbase[dl]);
  const float x1 = bf16_to_f32(kbase[dl + half]);
  const float kr = (d < half) ? (x0 * c - x1 * s) : (x0 * s + x1 * c);
  kc[((((long long)page * KVH + kvh) * (D / 8) + d / 8) * QSA_PAGE + pin) * 8 +
     d % 8] = f32_to_bf16(kr);
  vc[(((long long)page * KVH + kvh) * D + d) * QSA_PAGE + pin] =
      v[(long long)b * kvstride + (long long)kvh * D + d];
}

extern "C" void qsa_rope_kv_append_launch(
    unsigned short* q, const unsigned short* k, const unsigned short* v,
    unsigned short* kc, unsigned short* vc, const float* cos_t,
    const float* sin_t, const int* block_table, const int* seq_lens, int B,
    int QH, int KVH, int D, int max_pages, long long qstride,
    long long kvstride, hipStream_t stream) {
  hipLaunchKernelGGL(qsa_rope_kv_append, dim3(B * (QH + KVH)), dim3(D), 0,
                     stream, q, k, v, kc, vc, cos_t, sin_t, block_table,
                     seq_lens, B, QH, KVH, D, max_pages, qstride, kvstride);
}

// Un-fused single-step append (numerics tests / CPU-parity surface).
__global__ void
qsa_kv_append(const unsigned short* __restrict__ knew,  // [B, KVH, D]
              const unsigned short* __restrict__ vnew,
              unsigned short* __restrict__ kc, unsigned short* __restrict__ vc,
              const int* __restrict__ block_table, const int* __restrict__ seq_lens,
              int B, int KVH, int D, int max_pages, long long kvstride) {
  const int b = blockIdx.x / KVH;
  const int kvh = blockIdx.x % KVH;
  const int d = threadIdx.x;
  if (d >= D) return;
  const int pos = seq_lens[b] - 1;
  if (pos < 0) return;
  const int page = block_table[(long long)b * max_pages + pos / QSA_PAGE];
  const int pin = pos % QSA_PAGE;
  const unsigned short kv = knew[(long long)b * kvstride + (long long)kvh * D + d];
  const unsigned short vv = vnew[(long long)b * kvstride + (long long)kvh * D + d];
  kc[((((long long)page * KVH + kvh) * (D / 8) + d / 8) * QSA_PAGE + pin) * 8 +
     d % 8] = kv;
  vc[(((long long)page * KVH + kvh) * D + d) * QSA_PAGE + pin] = vv;
}

// Prefill bulk scatter: T tokens' k/v by precomputed slot ids
// (slot = page*64 + offset).  The V^T write is a 2-byte-per-thread scatter;
// consecutive tokens of a page share cache lines per d, so L2 absorbs it.
__global__ void
qsa_kv_scatter(const unsigned short* __restrict__ knew,  // [T, KVH, D] (row stride kvstride)
               const unsigned short* __restrict__ vnew,
               unsigned short* __restrict__ kc, unsigned short* __restrict__ vc,
               const int* __restrict__ slots,  // [T]
               int T, int KVH, int D, long long kvstride) {
  const long long t = blockIdx.x / KVH;
  const int kvh = blockIdx.x % KVH;
  const int d = threadIdx.x;
  if (t >= T || d >= D) return;
  const int slot = slots[t];
  const long long page = slot / QSA_PAGE;
  const int pin = slot % QSA_PAGE;
  const unsigned short kv = knew[t * kvstride + (long long)kvh * D + d];
  const unsigned short vv = vnew[t * kvstride + (long long)kvh * D + d];
  kc[(((page * KVH + kvh) * (D / 8) + d / 8) * QSA_PAGE + pin) * 8 + d % 8] = kv;
  vc[((page * KVH + kvh) * D + d) * QSA_PAGE + pin] = vv;
}

extern "C" void qsa_kv_append_launch(const unsigned short* knew,
                                     const unsigned short* vnew,
                                     unsigned short* kc, unsigned short* vc,
                                     const int* block_table,
                                     const int* seq_lens, int B, int KVH,
                                     int D, int max_pages, long long kvstride,
                                     hipStream_t stream) {
  hipLaunchKernelGGL(qsa_kv_append, dim3(B * KVH), dim3(D), 0, stream, knew,
                     vnew, kc, vc, block_table, seq_lens, B, KVH, D, max_pages,
                     kvstride);
}

extern "C" void qsa_kv_scatter_launch(const unsigned short* knew,
                                      const unsigned short* vnew,
                                      unsigned short* kc, unsigned short* vc,
                                      const int* slots, int T, int KVH, int D,
                                      long long kvstride, hipStream_t stream) {
  hipLaunchKernelGGL(qsa_kv_scatter, dim3((long long)T * KVH), dim3(D), 0,
                     stream, knew, vnew, kc, vc, slots, T, KVH, D, kvstride);
}

// ---------------------------------------------------------------------------
// Prefill rotation and cache write in one pass: q is rotated in place, or left for
// the attention to rotate (QH 0), k rotated on its way to the pages, v transposed into
// them through LDS.
//
// Block = (64 tokens, kv head): its R query heads, its key and its value.  A
// lane owns 8 dims and their rotation partners of one token, so angles are read
// once for all heads, and every access is 16 bytes wide; the page's K groups
// and V columns of neighbouring tokens lie together.  Bound by memory:
// 45k tokens, 32/8 heads of 128: 468 (rotation) + 292 us (scatter by elements)
// before, 224 us here (4.9 TB/s, what a copy reaches); few tokens are bound by
// round trips, so all reads of a pass come before its writes (5 tokens 6.8 -> 4.3
// us, 200 11.5 -> 6.1, 764 14.7 -> 7.8, the conversion's part among it).  The
// attention turns its queries in registers, so a prefill leaves q out: 10,528 tokens
// 51.7 -> 26.2 us, and the attention of 96 x 20-200 behind 500-1200 244 -> 254; 8192
// 41.6 -> 22.2, and 626 -> 614.
// ---------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(256)
qsa_rope_kv_scatter(unsigned short* __restrict__ q,        // [T, QH, D] strided
                    const unsigned short* __restrict__ k,  // [T, KVH, D]
                    const unsigned short* __restrict__ v,
                    unsigned short* __restrict__ kc,
                    unsigned short* __restrict__ vc,
                    const float* __restrict__ cos_t,
                    const float* __restrict__ sin_t,
                    const int* __restrict__ pos,           // [T]
                    const int* __restrict__ slots,         // [T], < 0: none
                    int T, int QH, int KVH, long long qstride,
                    long long kvstride) {
  constexpr int LT = D / 16;           // lanes per token
  constexpr int TB = 256 / LT;         // tokens per pass of the block
  constexpr int VP = D + 8;
  __shared__ __attribute__((aligned(16))) unsigned short vt[64 * VP];
  const int g = blockIdx.x % KVH;
  const long long t0 = (long long)(blockIdx.x / KVH) * 64;
  const int tid = threadIdx.x, R = QH / KVH;
  const int d = (tid % LT) * 8;
#pragma unroll
  for (int p = 0; p < 64; p += TB) {
    const int i = p + tid / LT;
    const long long t = t0 + i;
    if (t >= T) break;
    const long long at = (long long)pos[t] * (D / 2) + d;
    float c[8], s[8];
    ldv<float, 8>(cos_t + at, c);
    ldv<float, 8>(sin_t + at, s);
    // all reads before the first write: few tokens are a chain of latencies
    const int slot = slots[t];
    const long long row = t * kvstride + (long long)g * D + d;
    bf16x8_a kx = *reinterpret_cast<const bf16x8_a*>(k + row);
    bf16x8_a ky = *reinterpret_cast<const bf16x8_a*>(k + row + D / 2);
    const bf16x8_a vx = *reinterpret_cast<const bf16x8_a*>(v + row);
    const bf16x8_a vy = *reinterpret_cast<const bf16x8_a*>(v + row + D / 2);
    unsigned short* qp = q + t * qstride + (long long)g * R * D + d;
    for (int h = 0; h < R; h += 4, qp += 4 * D) {
      bf16x8_a x[4], y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (h + j < R) {
          x[j] = *reinterpret_cast<bf16x8_a*>(qp + j * D);
          y[j] = *reinterpret_cast<bf16x8_a*>(qp + j * D + D / 2);
        }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (h + j < R) {
          rotate_pair(x[j], y[j], c, s);
          *reinterpret_cast<bf16x8_a*>(qp + j * D) = x[j];
          *reinterpret_cast<bf16x8_a*>(qp + j * D + D / 2) = y[j];
        }
    }
    rotate_pair<true>(kx, ky, c, s);
    if (slot >= 0) {
      const long long tile =
          ((long long)(slot / QSA_PAGE) * KVH + g) * D * QSA_PAGE;
      unsigned short* kp =
          kc + tile + ((d / 8) * QSA_PAGE + slot % QSA_PAGE) * 8;
      *reinterpret_cast<bf16x8_a*>(kp) = kx;
      *reinterpret_cast<bf16x8_a*>(kp + D / 2 * QSA_PAGE) = ky;
    }
    *reinterpret_cast<bf16x8_a*>(vt + i * VP + d) = vx;
    *reinterpret_cast<bf16x8_a*>(vt + i * VP + d + D / 2) = vy;
  }
  __syncthreads();
  // lane = token: a wave's store is one column of the page's value tile
  const int lane = tid & 63;
  const long long t = t0 + lane;
  const int slot = t < T ? slots[t] : -1;
  if (slot < 0) return;
  unsigned short* vp =
      vc + ((long long)(slot / QSA_PAGE) * KVH + g) * D * QSA_PAGE +
      slot % QSA_PAGE;
#pragma unroll 8
  for (int e = tid >> 6; e < D; e += 4) vp[e * QSA_PAGE] = vt[lane * VP + e];
}

extern "C" void qsa_rope_kv_scatter_launch(
    unsigned short* q, const unsigned short* k, const unsigned short* v,
    unsigned short* kc, unsigned short* vc, const float* cos_t,
    const float* sin_t, const int* pos, const int* slots, int T, int QH,
    int KVH, int D, long long qstride, long long kvstride,
    hipStream_t stream) {
  const dim3 grid((unsigned)((long long)((T + 63) / 64) * KVH));
  if (D == 128)
    hipLaunchKernelGGL(qsa_rope_kv_scatter<128>, grid, dim3(256), 0, stream, q,
                       k, v, kc, vc, cos_t, sin_t, pos, slots, T, QH, KVH,
                       qstride, kvstride);
  else
    hipLaunchKernelGGL(qsa_rope_kv_scatter<64>, grid, dim3(256), 0, stream, q,
                       k, v, kc, vc, cos_t, sin_t, pos, slots, T, QH, KVH,
                       qstride, kvstride);
}

// ---------------------------------------------------------------------------
// Varlen flash PREFILL attention over the paged cache (K4 prefill path); with
// CAUSAL=false every row sees all keys of its item (the binding offers it; the
// encoder has a kernel of its own, encoder_attn.hip).
//
// Host passes maps of blocks of `rows` consecutive query tokens (item id,
// first token) plus per-item row offset / cached start / new length and the
// page table.
//
// Block = (token block, kv head): the R query heads of a kv head share its
// keys, so its tokens and heads together form the rows (row = token * R + head)
// of 16-row tiles, QT per wave, four waves.  Short portions thus fill tiles
// with heads, and K and V are read once per kv head.  Key heads run fastest
// over the blocks: with 8 of them a die's L2 keeps one.
// Scores come out transposed (row = key, column = query row): softmax state and
// rescale are lane-local, and the keys are dealt to the score tiles so that a
// lane ends up with 8 consecutive ones, which is the operand layout of the
// second product and of 16-byte V reads.  V's 16-byte groups are swizzled by
// row, so that 8 rows of a tile read all banks once.
//
// Each K and V page goes into LDS once per block, by loads that write it there
// in that order (the lanes' addresses are permuted, not the places), and both
// stand twice, so that a turn has one barrier: turn pg loads K of page pg + 2
// and V of page pg, and multiplies what came a turn before.  A page's products
// and its softmax depend on each other, and two blocks of a CU that stand at
// the same barriers do not fill each other's gaps, so a turn's softmax of page
// pg runs beside the products of page pg - 1 with its values, a few exponents
// and one fragment of V to each QT products, and the scores of page pg + 1
// follow, each fragment of K read PD - 1 ahead.  Maxima cross the groups of
// a column by lane swaps instead of the LDS crossbar.  The matrix cores are busy
// half of the time, the exponents a quarter; LDS reads (each K/V fragment
// serves QT tiles) take as long as the matrix cores.  Rescaling is left out when
// no maximum of the wave moved.
// Queries may be turned here, on their way into registers (what that saves stands at
// qsa_rope_kv_scatter): a row's dims d and d + D/2 are fragments of one lane.
// A wave's first and last page stand outside of the loop over the others: paths that
// meet behind the products took 30 registers more (D = 64: 149 us for 122).
// us, 32/8 heads of 128, with pages by way of registers and one after the other
// / here: 1 x 8192 tokens 643 / 533 (856 / 1032 TFLOP/s), 64 x 500-900 501 / 463,
// 96 x 20-200 behind 500-1200 293 / 256, 300 + 200 10.6 / 9.1; 16/8 heads, 8 x
// 1500-3000 206 / 175; 32/8 heads of 64, 32 x 500-900 130 / 124.
// ---------------------------------------------------------------------------
#define QSA_NEG (-3.0e38f)

template <int D, int QT, bool CAUSAL>
__global__ void __launch_bounds__(256, 2)
qsa_paged_attn_prefill(const unsigned short* __restrict__ q,   // [T, QH, D] strided
                       const unsigned short* __restrict__ kc,
                       const unsigned short* __restrict__ vc,
                       const int* __restrict__ block_table,    // [nb, npmax]
                       const int* __restrict__ qb_item,        // [QB]
                       const int* __restrict__ qb_pos0,        // [QB]
                       const int* __restrict__ item_off,       // [nb] row offset
                       const int* __restrict__ item_start,     // [nb] cached
                       const int* __restrict__ item_len,       // [nb] new rows
                       unsigned short* __restrict__ out,       // [T, QH*D]
                       float scale2, int QH, int KVH, int npmax,
                       long long qstride, int rows, int subs,
                       const float* __restrict__ cos_t,  // [positions, D/2], or
                       const float* __restrict__ sin_t,  // null: q is rotated
                       int positions) {
#ifdef __HIP_DEVICE_COMPILE__          // loads into LDS: not for the host
  constexpr int KS = D / 32;           // k-steps of a score tile
  constexpr int ET = D / 16;           // tiles of value columns
  constexpr int L = D / 32;            // 1 KB loads per wave, K and V each
  constexpr int PD = D == 64 ? 4 : 5;  // fragments of K or V in registers
  constexpr int TILE = QSA_PAGE * D;
  __shared__ __attribute__((aligned(16))) unsigned short kt[2 * TILE];
  __shared__ __attribute__((aligned(16))) unsigned short vt[2 * TILE];
  const int tid = threadIdx.x, lane = tid & 63;
  // a scalar: branches on it skip MFMAs, which ignore disabled lanes
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, hi = lane >> 4;
  const int R = QH / KVH;
  const int g = blockIdx.x % KVH;
  const int qb = blockIdx.x / KVH / subs, sub = blockIdx.x / KVH % subs;
  const int item = __builtin_amdgcn_readfirstlane(qb_item[qb]);
  const int pos0 = __builtin_amdgcn_readfirstlane(qb_pos0[qb]);
  const int n = __builtin_amdgcn_readfirstlane(item_len[item]);
  const int start = __builtin_amdgcn_readfirstlane(item_start[item]);
  const int v0 = pos0 * R + sub * 64 * QT;
  const int vend = min(pos0 + rows, n) * R;
  if (v0 >= vend) return;              // uniform over the block
  const long long off = item_off[item];
  // last key that any row of the block / of this wave sees
  const int last = __builtin_amdgcn_readfirstlane(
      start + (CAUSAL ? (min(v0 + 64 * QT, vend) - 1) / R : n - 1));
  const int w0 = v0 + wave * 16 * QT;
  const int wfirst = start + min(w0, vend - 1) / R;
  const int wlast = w0 >= vend ? -1
      : CAUSAL ? start + (min(w0 + 16 * QT, vend) - 1) / R : last;
  // pages of the block, those with keys for this wave, and those whose keys
  // all its rows see
  const int pages = last / QSA_PAGE + 1;
  const int mine =
      __builtin_amdgcn_readfirstlane(wlast < 0 ? 0 : wlast / QSA_PAGE + 1);
  const int whole = __builtin_amdgcn_readfirstlane(
      ((CAUSAL ? wfirst : last) + 1) / QSA_PAGE);

  // LDS places, in pieces of 16 bytes.  K [D/8][64 keys]: place p of a row holds
  // the key that row p % 16 of score tile p / 16 stands for, 32s + 8h + 4t + r in
  // row 4h + r of tile 2s + t.  V [D][8]: group j of 8 keys of column e stands
  // at j ^ sw(e), sw = e&3 | (e>>3 & 1) << 2.  A load fills 1 KB in the order of
  // the lanes: one row of K, 8 columns of V.
  const unsigned kfrom = wave * 1024 + ((lane >> 5) * 32 + (lane >> 2 & 3) * 8 +
                                        (lane >> 4 & 1) * 4 + (lane & 3)) * 16;
  const unsigned vfrom = wave * 1024 + (lane >> 3) * 128 +
      ((lane & 7) ^ ((lane >> 3 & 3) | (wave & 1) << 2)) * 16;
  const auto table = (const __attribute__((address_space(4))) int*)(
      block_table + (long long)item * npmax);
  auto load = [&](const unsigned short* cache, unsigned short* to, int pg,
                  unsigned from) __attribute__((always_inline)) {
    const long long tile = ((long long)table[pg] * KVH + g) * TILE;
    const __amdgpu_buffer_rsrc_t page = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(cache + tile), 0, TILE * 2, 0x00027000);
#pragma unroll
    for (int i = 0; i < L; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          page, (__attribute__((address_space(3))) void*)(
                    to + (pg & 1) * TILE + (wave + 4 * i) * 512),
          16, from, i * 4096, 0, 0);
  };
  // all that the waves loaded has arrived, and they have read what they wanted
  auto arrived = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(7 << 4);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  load(kc, kt, 0, kfrom);
  if (pages > 1) load(kc, kt, 1, kfrom);

  // maxima are taken before the scale, which therefore has to be positive
  const bool negative = scale2 < 0.f;
  scale2 = fmaxf(fabsf(scale2), 1e-30f);
  bf16x8_v qf[QT][KS];
  int qpos[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    const int v = min(w0 + u * 16 + col, vend - 1);
    const int tok = v / R;
    qpos[u] = CAUSAL ? start + tok : last;
    const unsigned short* qrow =
        q + (off + tok) * qstride + (long long)(g * R + v - tok * R) * D;
#pragma unroll
    for (int s = 0; s < KS; ++s)
      qf[u][s] = *reinterpret_cast<const bf16x8_v*>(qrow + s * 32 + hi * 8);
  }
  if (cos_t) {                         // dims d and d + D/2 are a lane's
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      const int tok = min(w0 + u * 16 + col, vend - 1) / R;
      const long long at =
          (long long)min(start + tok, positions - 1) * (D / 2) + hi * 8;
#pragma unroll
      for (int s = 0; s < KS / 2; ++s) {
        float c[8], sn[8];
        ldv<float, 8>(cos_t + at + s * 32, c);
        ldv<float, 8>(sin_t + at + s * 32, sn);
        rotate_pair(qf[u][s], qf[u][s + KS / 2], c, sn);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < QT; ++u)
#pragma unroll
    for (int s = 0; s < KS; ++s)
      if (negative) qf[u][s] ^= (short)0x8000;
  f32x4_v acc[QT][ET], sc[QT][4];
  bf16x8_v pf[QT][2];
  float m[QT], l[QT], alpha[QT], psum[QT], top[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    m[u] = QSA_NEG;
    l[u] = 0.f;
    alpha[u] = 1.f;
#pragma unroll
    for (int t = 0; t < ET; ++t) acc[u][t] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  }
  bool moved = false;                  // a maximum, by the last softmax

  // fragment c of a page: keys of tile c % 4, k-step c / 4; row i of tile t of
  // the values is column 32(t/2) + 8(i/4) + 4(t%2) + i%4, so that a lane
  // collects 8 consecutive columns over two tiles
  auto keys = [&](const unsigned short* k, int c) __attribute__((always_inline)) {
    return *reinterpret_cast<const bf16x8_v*>(
        k + (((c >> 2) * 4 + hi) * 64 + (c & 3) * 16 + col) * 8);
  };
  const int vrow = (col >> 2) * 8 + (col & 3);
  auto vals = [&](const unsigned short* v, int c) __attribute__((always_inline)) {
    const int s = c / ET, t = c % ET;
    const int e = (t >> 1) * 32 + (t & 1) * 4 + vrow;
    return *reinterpret_cast<const bf16x8_v*>(
        v + (e * 8 + ((s * 4 + hi) ^ (col & 7))) * 8);
  };
  auto scores = [&](const unsigned short* k) __attribute__((always_inline)) {
    bf16x8_v f[PD];
#pragma unroll
    for (int c = 0; c < PD - 1; ++c) f[c] = keys(k, c);
#pragma unroll
    for (int c = 0; c < 4 * KS; ++c) {
      __builtin_amdgcn_sched_barrier(0);
      if (c + PD - 1 < 4 * KS) f[(c + PD - 1) % PD] = keys(k, c + PD - 1);
#pragma unroll
      for (int u = 0; u < QT; ++u)
        sc[u][c & 3] = mfma_bf16(
            f[c % PD], qf[u][c >> 2],
            c < 4 ? (f32x4_v){0.f, 0.f, 0.f, 0.f} : sc[u][c & 3]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto maximum = [&](int u) __attribute__((always_inline)) {
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[u][i >> 2][i & 3]);
    top[u] = fmaxf(m[u], rows_max(mx) * scale2);
    moved |= top[u] > m[u];
    alpha[u] = __builtin_amdgcn_exp2f(m[u] - top[u]);
    psum[u] = 0.f;
  };
  unsigned int pk[QT][8];
  auto weights = [&](int u, int j) __attribute__((always_inline)) {
    const float a = __builtin_amdgcn_exp2f(
        fmaf(sc[u][j >> 1][(j & 1) * 2], scale2, -top[u]));
    const float b = __builtin_amdgcn_exp2f(
        fmaf(sc[u][j >> 1][(j & 1) * 2 + 1], scale2, -top[u]));
    psum[u] += a;
    psum[u] += b;
    pk[u][j] = cvt_bf16x2(a, b);
  };
  auto packed = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < QT; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        pf[u][s] = __builtin_bit_cast(
            bf16x8_v, make_uint4(pk[u][4 * s], pk[u][4 * s + 1],
                                 pk[u][4 * s + 2], pk[u][4 * s + 3]));
  };
  // softmax of sc by itself; a NaN score counts as no key
  auto guarded = [&]() __attribute__((always_inline)) {
    moved = false;
#pragma unroll
    for (int u = 0; u < QT; ++u) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        sc[u][i >> 2][i & 3] = fmaxf(sc[u][i >> 2][i & 3], -INFINITY);
      maximum(u);
#pragma unroll
      for (int j = 0; j < 8; ++j) weights(u, j);
    }
    packed();
  };
  // softmax of sc beside the products of the weights before it with v; the
  // first QT chunks take the maxima, the rest share the exponents
  auto beside = [&](const unsigned short* v) __attribute__((always_inline)) {
    constexpr int NC = ET * 2, PAIRS = QT * 8, SPAN = NC - 2;
    bf16x8_v f[PD];
    moved = false;
#pragma unroll
    for (int c = 0; c < PD - 1; ++c) f[c] = vals(v, c);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      __builtin_amdgcn_sched_barrier(0);
      if (c + PD - 1 < NC) f[(c + PD - 1) % PD] = vals(v, c + PD - 1);
#pragma unroll
      for (int u = 0; u < QT; ++u)
        acc[u][c % ET] = mfma_bf16(f[c % PD], pf[u][c / ET], acc[u][c % ET]);
      if (c < QT) maximum(c);
#pragma unroll
      for (int i = 0; i < PAIRS; ++i)
        if (c == 2 + i * SPAN / PAIRS) weights(i >> 3, i & 7);
    }
    __builtin_amdgcn_sched_barrier(0);
    packed();
  };

  // a turn's barrier and loads: K of page pg + 1 and V of pg - 1 are there
  auto stage = [&](int pg) __attribute__((always_inline)) {
    arrived();
    if (pg + 2 < pages) load(kc, kt, pg + 2, kfrom);
    if (pg < pages) {
      load(vc, vt, pg, vfrom);
      return;
    }
    const int have = last - (pg - 1) * QSA_PAGE;  // keys 0..have count
    if (have == QSA_PAGE - 1) return;
    // slots nobody has written yet may hold anything, NaN too
    unsigned short* v = vt + ((pg + 1) & 1) * TILE;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int at = tid + i * 256, e = at >> 3;
      const int k0 = ((at & 7) ^ ((e & 3) | (e >> 1 & 4))) * 8;
      u32x4_v x = *reinterpret_cast<u32x4_v*>(v + at * 8);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = k0 + 2 * c;
        x[c] = k > have ? 0u : k + 1 > have ? x[c] & 0xffffu : x[c];
      }
      *reinterpret_cast<u32x4_v*>(v + at * 8) = x;
    }
    lds_barrier();
  };
  // keys of page pg that a row does not see
  auto hide = [&](int pg) __attribute__((always_inline)) {
    if (pg < whole) return;
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      const int see = qpos[u] - pg * QSA_PAGE - hi * 8;
#pragma unroll
      for (int pt = 0; pt < 4; ++pt) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if ((pt >> 1) * 32 + (pt & 1) * 4 + r > see) sc[u][pt][r] = -INFINITY;
        __builtin_amdgcn_sched_barrier(0);  // few masks at a time
      }
    }
  };
  auto advance = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      m[u] = top[u];
      l[u] = l[u] * alpha[u] + psum[u];
    }
  };
  auto rescale = [&]() __attribute__((always_inline)) {
    if (!__any(moved)) return;         // every factor is 1
#pragma unroll
    for (int u = 0; u < QT; ++u)
#pragma unroll
      for (int t = 0; t < ET; ++t) acc[u][t] *= alpha[u];
  };

  arrived();
  if (mine > 0) scores(kt);
  stage(0);
  int pg = 1;
  if (mine > 0) {
    hide(0);
    guarded();
    advance();
    moved = false;                     // there is nothing to rescale yet
    if (mine > 1) scores(kt + TILE);
#pragma clang loop unroll(disable)
    for (; pg < mine; ++pg) {
      stage(pg);
      const int other = ((pg + 1) & 1) * TILE;
      rescale();
      hide(pg);
      beside(vt + other);
      bool bad = false;
#pragma unroll
      for (int u = 0; u < QT; ++u) bad |= !(psum[u] <= 64.f);
      if (__any(bad)) guarded();       // masked scores are -inf by now
      advance();
      if (pg + 1 < mine) scores(kt + other);
    }
    stage(pg);
    rescale();
    const unsigned short* v = vt + ((pg + 1) & 1) * TILE;
#pragma unroll
    for (int c = 0; c < 2 * ET; ++c) {
      const bf16x8_v a = vals(v, c);
#pragma unroll
      for (int u = 0; u < QT; ++u)
        acc[u][c % ET] = mfma_bf16(a, pf[u][c / ET], acc[u][c % ET]);
      if (c & 1) __builtin_amdgcn_sched_barrier(0);
    }
    ++pg;
  }
#pragma clang loop unroll(disable)
  for (; pg <= pages; ++pg) stage(pg);

#pragma unroll
  for (int u = 0; u < QT; ++u) {
    l[u] = rows_sum(l[u]);
    const float inv = l[u] > 0.f ? 1.f / l[u] : 0.f;
    const int v = w0 + u * 16 + col;
    if (v >= vend) continue;
    const int tok = v / R;
    unsigned short* orow = out + (off + tok) * ((long long)QH * D) +
                           (long long)(g * R + v - tok * R) * D;
#pragma unroll
    for (int t = 0; t < ET; t += 2) {
      const f32x4_v a = acc[u][t] * inv, b = acc[u][t + 1] * inv;
      *reinterpret_cast<uint4*>(orow + t * 16 + hi * 8) =
          make_uint4(cvt_bf16x2(a[0], a[1]), cvt_bf16x2(a[2], a[3]),
                     cvt_bf16x2(b[0], b[1]), cvt_bf16x2(b[2], b[3]));
    }
  }
#endif
}

extern "C" void qsa_paged_attn_prefill_launch(
    const unsigned short* q, const unsigned short* kc,
    const unsigned short* vc, const int* block_table, const int* qb_item,
    const int* qb_pos0, const int* item_off, const int* item_start,
    const int* item_len, unsigned short* out, float scale, int QB, int QH,
    int KVH, int npmax, int D, long long qstride, int causal, int rows,
    const float* cos_t, const float* sin_t, int positions,
    hipStream_t stream) {
  const float scale2 = scale * 1.4426950408889634f;
  // two tiles per wave as soon as a block's rows fill more than one each
  const int vrows = rows * (QH / KVH), qt = vrows > 64 ? 2 : 1;
  const int subs = (vrows + 64 * qt - 1) / (64 * qt);
  const dim3 grid((unsigned)((long long)QB * KVH * subs));
  if (grid.x == 0) return;
#define QSA_PREFILL_CASE(DD, QQ, CC)                                          \
  if (D == DD && qt == QQ && causal == (int)CC) {                             \
    hipLaunchKernelGGL((qsa_paged_attn_prefill<DD, QQ, CC>), grid, dim3(256), \
                       0, stream, q, kc, vc, block_table, qb_item, qb_pos0,   \
                       item_off, item_start, item_len, out, scale2, QH, KVH,  \
                       npmax, qstride, rows, subs, cos_t, sin_t, positions);  \
    return;                                                                   \
  }
  QSA_PREFILL_CASE(128, 1, true) QSA_PREFILL_CASE(128, 1, false)
  QSA_PREFILL_CASE(64, 1, true) QSA_PREFILL_CASE(64, 1, false)
  QSA_PREFILL_CASE(128, 2, true) QSA_PREFILL_CASE(128, 2, false)
  QSA_PREFILL_CASE(64, 2, true) QSA_PREFILL_CASE(64, 2, false)
#undef QSA_PREFILL_CASE
}
