// GPU hash join for streaming enrichment (K8):
// build a latest-row-per-key hash table from a dimension batch in HBM,
// probe it with a stream batch, TTL-filter at probe time.
//
// Semantics match runtime/joins.TTLTable + enrich_join (the reference's
// `orders JOIN customers JOIN products` under SET 'sql.state-ttl',
// LAB1-Walkthrough.md:119-131): keys are pre-hashed to i64 on the host
// (columnar batches from the Avro codec), the table keeps the row with
// the LATEST event time per key, and a probe returns that row's index or
// -1 if absent/expired.
//
// Table layout: open addressing, power-of-two capacity, a key's slots an odd
// step of its own hash apart (qsa_hj_slots).
//   slot = {key u64, pay u64}: key EMPTY = 0xFFFFFFFFFFFFFFFF (hashed keys
//                never collide with it: host masks hashes to 63 bits), pay
//                packed (ts << 24) | row  — one atomicMax keeps the
//                latest-ts row per key (row < 2^24, ts < 2^40 ms ≈ 34 y)
// Both words of a slot lie in one cache line, so a probe is one 16-byte load
// where separate key and payload arrays take two dependent ones; the probes of
// a wave hit 64 different lines and that access rate is what bounds them.
// 2M probes of a 50,000-row table: 27 us with separate arrays, 18 us here.
// (The bindings hand the two words out as strided views; STRIDE 1 serves
// tables held as two arrays.)
// Insert: atomicCAS on the key slots in turn, then atomicMax on the payload.  No
// locks, no host round trips; eviction is at probe time (ts >= cutoff), full
// compaction = rebuild from the surviving rows.
#include "common.h"

#define QSA_HJ_EMPTY 0xFFFFFFFFFFFFFFFFull

__device__ __forceinline__ unsigned long long qsa_hj_mix(
    unsigned long long x) {
  // splitmix64 finalizer: spreads host hashes over the table
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// Where a key is looked for.  Neighbours in the table would form runs, whose
// longest is what a build waits for, an atomic access to memory per slot: 50,000
// rows 13.1 us with steps of one, 10 to 12 so, 2M probes of them 19.8 and 17 to 18,
// 500k 8.7 and 7.  A table beyond a die's L2 (4 MiB) has steps of one, whose next
// slot mostly lies in the line that has come (2M probes of 1M rows 43.5 us, 50.3
// with others).
#define QSA_HJ_NEAR (1u << 18)         // slots

struct QsaSlots {
  unsigned int at, step;
};

__device__ __forceinline__ QsaSlots qsa_hj_slots(unsigned long long key,
                                                 unsigned int mask) {
  const unsigned long long h = qsa_hj_mix(key);
  return {(unsigned int)h & mask,
          mask < QSA_HJ_NEAR ? (unsigned int)(h >> 32) | 1u : 1u};
}

__global__ void qsa_hash_clear(ulonglong2* __restrict__ slots, int cap) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cap) slots[i] = make_ulonglong2(QSA_HJ_EMPTY, 0ull);
}

__global__ void qsa_hash_build(const long long* __restrict__ keys,   // [N]
                               const long long* __restrict__ ts,     // [N]
                               unsigned long long* __restrict__ slots,
                               int n, unsigned int mask) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned long long key = (unsigned long long)keys[i];
  // event times clamp to the 40 bits the payload has for them
  const long long t = min(max(ts[i], 0ll), (1ll << 40) - 1);
  const unsigned long long pay =
      (((unsigned long long)t) << 24) | (unsigned int)(i & 0xFFFFFF);
  QsaSlots s = qsa_hj_slots(key, mask);
  for (unsigned int probe = 0; probe <= mask; ++probe) {
    unsigned long long prev =
        atomicCAS(&slots[2ull * s.at], QSA_HJ_EMPTY, key);
    if (prev == QSA_HJ_EMPTY || prev == key) {
      atomicMax(&slots[2ull * s.at + 1], pay);   // latest event time wins
      return;
    }
    s.at = (s.at + s.step) & mask;
  }
  // table full: drop (host sizes cap >= 2*n, unreachable)
}

template <int STRIDE>                  // words between slots
__global__ void __launch_bounds__(256)
qsa_hash_probe(const long long* __restrict__ keys,   // [M]
               const unsigned long long* __restrict__ tkeys,
               const unsigned long long* __restrict__ tpay,
               int* __restrict__ out_row,            // [M]
               int m, unsigned int mask, long long min_ts) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= m) return;
  const unsigned long long key = (unsigned long long)keys[i];
  QsaSlots s = qsa_hj_slots(key, mask);
  int row = -1;
  for (unsigned int probe = 0; probe <= mask; ++probe) {
    unsigned long long k, pay;
    if constexpr (STRIDE == 2) {
      const ulonglong2 both =
          reinterpret_cast<const ulonglong2*>(tkeys)[s.at];
      k = both.x;
      pay = both.y;
    } else {
      k = tkeys[s.at];
      pay = tpay[s.at];
    }
    if (k == QSA_HJ_EMPTY) break;
    if (k == key) {
      if ((long long)(pay >> 24) >= min_ts) row = (int)(pay & 0xFFFFFF);
      break;
    }
    s.at = (s.at + s.step) & mask;
  }
  out_row[i] = row;
}

extern "C" void qsa_hash_build_launch(const long long* keys,
                                      const long long* ts,
                                      unsigned long long* slots, int n,
                                      unsigned int mask,
                                      hipStream_t stream) {
  const int bs = 256, cap = (int)mask + 1;
  hipLaunchKernelGGL(qsa_hash_clear, dim3((cap + bs - 1) / bs), dim3(bs), 0,
                     stream, reinterpret_cast<ulonglong2*>(slots), cap);
  if (n == 0) return;
  hipLaunchKernelGGL(qsa_hash_build, dim3((n + bs - 1) / bs), dim3(bs), 0,
                     stream, keys, ts, slots, n, mask);
}

extern "C" void qsa_hash_probe_launch(const long long* keys,
                                      const unsigned long long* tkeys,
                                      const unsigned long long* tpay,
                                      int* out_row, int m, unsigned int mask,
                                      long long min_ts, int paired,
                                      hipStream_t stream) {
  if (m == 0) return;
  const dim3 grid((unsigned)(((long long)m + 255) / 256));
  if (paired)
    hipLaunchKernelGGL(qsa_hash_probe<2>, grid, dim3(256), 0, stream, keys,
                       tkeys, tpay, out_row, m, mask, min_ts);
  else
    hipLaunchKernelGGL(qsa_hash_probe<1>, grid, dim3(256), 0, stream, keys,
                       tkeys, tpay, out_row, m, mask, min_ts);
}
