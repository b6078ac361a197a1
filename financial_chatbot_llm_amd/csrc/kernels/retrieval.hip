// K15: filtered exact top-k similarity search over an HBM-resident corpus (replaces Qdrant's
// filtered HNSW query, tools/qdrant_tool.py:98-153).
//
// Filters are the reference's: user_id == u (always) AND date >= t (optional).  Such filters are
// very selective (one user's rows out of ~1M), so the search is organised around the filter, not
// the vectors:
//   1. filter_compact: one pass over the int32 user codes (and, near a match, the int64 dates)
//      evaluates every query's filter and appends matching row ids to a per-query
//      candidate list (wave-aggregated atomics).  Vectors of non-matching rows are never read.
//   2. rank: waves compute <corpus_row, query> of the candidate rows (768-d bf16, 16 B/lane), and one
//      workgroup per query ranks up to SORT_CAP (score, row) pairs in LDS, descending by score, ties by
//      row id, and writes the first k.
// Queries with more candidates than SORT_CAP are finished by the caller (torch.topk on the
// device-side score list), which the host detects from the returned counts.
#include "common.h"

#define SORT_CAP 8192
#define CSTRIDE 32      // counters lie a cache line apart: beside each other, their atomics wait for one another

// A block takes FROWS * 256 rows at a time, a thread FROWS of them, 256 apart; the codes and the queries are fetched together.
// The first look at the codes only finds the queries that a row of the wave belongs to (seldom more than one); the dates are read
// for waves with any, and the append is made for those queries.  Bound by that chain: codes, dates, counter, list.  1M rows, 16
// queries, the codes in the caches from a search before: 6 us; every query of a wave with a hit looked at again 11, dates always read and
// counters side by side 14.
constexpr int FROWS = 2;
__global__ void __launch_bounds__(256) filter_compact_kernel(const int* __restrict__ user_codes,
                                                             const long long* __restrict__ dates, long N,
                                                             const int* __restrict__ q_user,
                                                             const long long* __restrict__ q_floor, int nq,
                                                             int* __restrict__ counts, int* __restrict__ cand, int cap) {
  __shared__ __attribute__((aligned(16))) int su[64];
  __shared__ long long sf[64];
  const int lane = threadIdx.x & 63;
  bool first = true;
  for (long base = (long)blockIdx.x * (256 * FROWS); base < N; base += (long)gridDim.x * (256 * FROWS)) {
    int code[FROWS];
    bool in[FROWS];
#pragma unroll
    for (int r = 0; r < FROWS; ++r) {
      const long n = base + 256 * r + threadIdx.x;
      in[r] = n < N;
      code[r] = user_codes[in[r] ? n : N - 1];
    }
    if (first) {
      if (threadIdx.x < 64) {                              // beyond the queries the last one again
        const int q = min((int)threadIdx.x, nq - 1);
        su[threadIdx.x] = q_user[q];
        sf[threadIdx.x] = q_floor[q];
      }
      __syncthreads();
      first = false;
    }
    unsigned long long present = 0;
    for (int q = 0; q < nq; q += 4) {
      const int4 u = *reinterpret_cast<const int4*>(su + q);
      bool h[4] = {};
#pragma unroll
      for (int r = 0; r < FROWS; ++r) h[0] |= code[r] == u.x, h[1] |= code[r] == u.y, h[2] |= code[r] == u.z, h[3] |= code[r] == u.w;
#pragma unroll
      for (int i = 0; i < 4; ++i) present |= (unsigned long long)(__ballot(h[i]) != 0) << (q + i);
    }
    if (nq < 64) present &= (1ull << nq) - 1;
    if (!present) continue;
    long long d[FROWS];
#pragma unroll
    for (int r = 0; r < FROWS; ++r) d[r] = dates[in[r] ? base + 256 * r + threadIdx.x : N - 1];
    auto matches = [&](int qi, unsigned long long (&mask)[FROWS]) {
      const int u = su[qi];
      const long long since = sf[qi];
      int hits = 0;
#pragma unroll
      for (int r = 0; r < FROWS; ++r) {
        mask[r] = __ballot(in[r] && code[r] == u && d[r] >= since);
        hits += __popcll(mask[r]);
      }
      return hits;
    };
    unsigned long long mask[FROWS], left = present;
    int mine = 0, start = 0;                               // of query `lane`: one trip for the counters of all
    for (; left; left &= left - 1) {
      const int qi = __ffsll(left) - 1, hits = matches(qi, mask);
      if (hits == 0) present &= ~(1ull << qi);
      if (lane == qi) mine = hits;
    }
    if (mine) start = atomicAdd(&counts[lane * CSTRIDE], mine);
    for (; present; present &= present - 1) {
      const int qi = __ffsll(present) - 1;
      matches(qi, mask);
      int at = __shfl(start, qi, 64);
#pragma unroll
      for (int r = 0; r < FROWS; ++r) {
        const int pos = at + __popcll(mask[r] & ((1ull << lane) - 1ull));
        if ((mask[r] >> lane & 1) && pos < cap) cand[(long)qi * cap + pos] = (int)(base + 256 * r + threadIdx.x);
        at += __popcll(mask[r]);
      }
    }
  }
}

__device__ __forceinline__ bool before(float sa, int ia, float sb, int ib) {  // a ranks before b
  return sa > sb || (sa == sb && ia < ib);
}

// The first k of cnt <= 1024 E scored rows, by 1024 threads with E neighbouring places of the sorting network each: partners in the
// same thread are compared in registers, those of a wave by lane exchange, and only the widest strides go through LDS with a barrier
// (10 of 78 steps for 4096 rows).  One query of 3300 rows, scored
// and ranked: 32 us, with all steps through LDS 97.  A row's key is its score, turned so that whole numbers
// ascend as scores descend, and its id; scores that are not numbers come last.
template <int E>
__device__ __forceinline__ void sort_first(const float* __restrict__ scores, const int* __restrict__ ids, int cnt, int k, uint64_t* lds,
                                           int* __restrict__ out_ids, float* __restrict__ out_scores) {
  const int t = threadIdx.x;
  uint64_t key[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = t * E + e;
    key[e] = ~0ull;
    if (i < cnt) {
      const float s = scores[i] + 0.f;                     // (-0 is 0)
      const unsigned u = __float_as_uint(s), down = u >> 31 ? u : ~u & 0x7fffffffu;
      key[e] = (uint64_t)(s == s ? down : 0xffffffffu) << 32 | (unsigned)ids[i];
    }
  }
  for (int size = 2; size <= 1024 * E; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= E) {
        const int far = stride / E;                        // threads between partners
        const bool low = ((t & far) == 0) == ((t & (size / E)) == 0);
        uint64_t other[E];
        if (far >= 64) {
          __syncthreads();
#pragma unroll
          for (int e = 0; e < E; ++e) lds[e * 1024 + t] = key[e];
          __syncthreads();
#pragma unroll
          for (int e = 0; e < E; ++e) other[e] = lds[e * 1024 + (t ^ far)];
        } else {
#pragma unroll
          for (int e = 0; e < E; ++e) other[e] = __shfl_xor((unsigned long long)key[e], far, 64);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) key[e] = (other[e] < key[e]) == low ? other[e] : key[e];
      } else {
#pragma unroll
        for (int s = E / 2; s > 0; s >>= 1)
          if (s == stride) {
#pragma unroll
            for (int e = 0; e < E; ++e)
              if ((e & s) == 0) {
                const bool up = ((t * E + e) & size) == 0;
                if ((key[e + s] < key[e]) == up) {
                  const uint64_t x = key[e];
                  key[e] = key[e + s];
                  key[e + s] = x;
                }
              }
          }
      }
    }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = t * E + e;
    const unsigned down = key[e] >> 32;
    if (i < k) {
      out_ids[i] = (int)(unsigned)key[e];
      out_scores[i] = __uint_as_float(down >> 31 ? down : ~down & 0x7fffffffu);
    }
  }
}

// gridDim.x blocks per query: the scores of its candidates, the first k of them, -1 / 0 behind those, the count to the device and
// (host_count) to the host, and the counters back to zero for the next call.  Up to ALONE candidates the query's first block scores
// and ranks them by itself, SROWS rows a wave in flight; of more, every block scores a share and the last one to be done ranks
// them: it has drawn the last of the query's tickets, behind which the others' scores have left their caches.  D a multiple of 8 up to 1024.
// Ranking: up to RANK_CAP candidates each finds its rank by counting those before it, 1024 threads over all pairs; more are sorted (28
// barriers).  16 queries of about 90: 7 us in one launch; scores and ranks in a launch each 3.6 and 6.8 with 1.2 between.
constexpr int RANK_CAP = 256, ALONE = 128, SROWS = 4;
__global__ void __launch_bounds__(1024) rank_kernel(const bf16* __restrict__ corpus, int D, const bf16* __restrict__ queries,
                                                    int* __restrict__ counts, const int* __restrict__ cand, float* scores, int cap,
                                                    const int* __restrict__ ks, int kmax, int* __restrict__ out_ids,
                                                    float* __restrict__ out_scores, int* __restrict__ out_count,
                                                    int* __restrict__ host_count) {
  extern __shared__ __attribute__((aligned(16))) char dyn[];
  float* ss = reinterpret_cast<float*>(dyn);
  int* si = reinterpret_cast<int*>(dyn + SORT_CAP * sizeof(float));
  __shared__ int rank[RANK_CAP];
  __shared__ int last;
  const int qi = blockIdx.y, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int total = counts[qi * CSTRIDE];
  const int cnt = min(total, cap);
  const bool big = total > SORT_CAP;                       // the host finishes this query
  const bool alone = cnt <= ALONE;
  const int k = big ? 0 : min(ks[qi], min(cnt, kmax));
  if (!alone || blockIdx.x == 0) {
    const int nch = D >> 3, waves = alone ? 16 : 16 * gridDim.x;
    float qv[2][8];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int c = lane + 64 * r;
      if (c < nch) unpack8(reinterpret_cast<const uint4*>(queries + (long)qi * D)[c], qv[r]);
    }
    for (int i = alone ? w : blockIdx.x * 16 + w; i < cnt; i += SROWS * waves) {
      int row[SROWS];
      uint4 v[SROWS][2];
#pragma unroll
      for (int j = 0; j < SROWS; ++j) row[j] = cand[(long)qi * cap + min(i + j * waves, cnt - 1)];
      if (nch > 0) {
#pragma unroll
        for (int j = 0; j < SROWS; ++j)
#pragma unroll
          for (int r = 0; r < 2; ++r)
            v[j][r] = reinterpret_cast<const uint4*>(corpus + (long)row[j] * D)[min(lane + 64 * r, nch - 1)];
      }
#pragma unroll
      for (int j = 0; j < SROWS; ++j) {
        float acc = 0.f;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          if (lane + 64 * r < nch) {
            float f[8];
            unpack8(v[j][r], f);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc += f[e] * qv[r][e];
          }
        }
        acc = wave_sum(acc);
        const int at = i + j * waves;
        if (lane == 0 && at < cnt) {
          if (alone) ss[at] = acc, si[at] = row[j];
          else scores[(long)qi * cap + at] = acc;
        }
      }
    }
  }
  for (int i = max(k, 0) + blockIdx.x * 1024 + threadIdx.x; i < kmax; i += gridDim.x * 1024) {
    out_ids[(long)qi * kmax + i] = -1;
    out_scores[(long)qi * kmax + i] = 0.f;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();                                         // the block has read the count and written its scores
  if (threadIdx.x == 0) {
    if (!alone) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    last = __hip_atomic_fetch_add(&counts[qi * CSTRIDE + 1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    if (last) {
      if (!alone) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      counts[qi * CSTRIDE] = 0;
      counts[qi * CSTRIDE + 1] = 0;
    }
  }
  if (threadIdx.x < RANK_CAP) rank[threadIdx.x] = 0;
  __syncthreads();
  if (alone ? blockIdx.x != 0 : !last) return;
  if (threadIdx.x == 0) {
    out_count[qi] = big ? -total : k;
    if (host_count != nullptr) host_count[qi] = big ? -total : k;
  }
  if (big || cnt == 0) return;
  if (cnt > RANK_CAP) {
    uint64_t* keys = reinterpret_cast<uint64_t*>(dyn);
    const float* sc = scores + (long)qi * cap;
    const int* id = cand + (long)qi * cap;
    int* oi = out_ids + (long)qi * kmax;
    float* os = out_scores + (long)qi * kmax;
    if (cnt <= 1024) sort_first<1>(sc, id, cnt, k, keys, oi, os);
    else if (cnt <= 2048) sort_first<2>(sc, id, cnt, k, keys, oi, os);
    else if (cnt <= 4096) sort_first<4>(sc, id, cnt, k, keys, oi, os);
    else sort_first<8>(sc, id, cnt, k, keys, oi, os);
    return;
  }
  if (!alone) {
    if (threadIdx.x < cnt) {
      ss[threadIdx.x] = scores[(long)qi * cap + threadIdx.x];
      si[threadIdx.x] = cand[(long)qi * cap + threadIdx.x];
    }
    __syncthreads();
  }
  int n = 1;
  while (n < cnt) n <<= 1;
  const int i = threadIdx.x % n, part = threadIdx.x / n, parts = 1024 / n;
  if (i < cnt) {
    auto key = [&](int x) { return ss[x] == ss[x] ? ss[x] : -INFINITY; };   // a total order: no rank is left out
    const float s = key(i);
    const int id = si[i];
    int r = 0;
    for (int j = part; j < cnt; j += parts) r += before(key(j), si[j], s, id);
    atomicAdd(&rank[i], r);
  }
  __syncthreads();
  if (threadIdx.x < cnt && rank[threadIdx.x] < k) {
    out_ids[(long)qi * kmax + rank[threadIdx.x]] = si[threadIdx.x];
    out_scores[(long)qi * kmax + rank[threadIdx.x]] = ss[threadIdx.x];
  }
}

// The candidates of every query.  counts [nq][32] (number and tickets): zero at the first call, zero again behind every pair of
// calls; cand [nq][cap].  Everything penny_topk_rank refuses is refused here, before the counters move.
PENNY_API int penny_topk_filter(const int* user_codes, const long long* dates, long N, int D, const int* q_user,
                                const long long* q_floor, int nq, int* counts, int* cand, int cap, hipStream_t stream) {
  if (nq <= 0) return 0;
  if (nq > 64 || D % 8 || D > 1024) return (int)hipErrorInvalidValue;
  long g = (N + 256 * FROWS - 1) / (256 * FROWS);
  if (g > 4096) g = 4096;
  if (g < 1) g = 1;
  hipLaunchKernelGGL(filter_compact_kernel, dim3((int)g), dim3(256), 0, stream, user_codes, dates, N, q_user, q_floor,
                     nq, counts, cand, cap);
  PENNY_RETURN_LAUNCH();
}

// Their first k, behind penny_topk_filter of the same lists.  host_count (pinned host memory, or null): out_count as well, and the
// call returns when all of it is done: a caller may read the results on any stream.  (Going on as soon as the counts are known saves 12 us
// between calls whose results nobody reads, 3 us where they are read, and leaves the ranking to run behind the return.)
PENNY_API int penny_topk_rank(const void* corpus, int D, const void* queries, const int* ks, int nq, int kmax, int* counts,
                              const int* cand, float* scores, int cap, int* out_ids, float* out_scores, int* out_count,
                              int* host_count, hipStream_t stream) {
  if (nq <= 0) return 0;
  if (nq > 64 || D % 8 || D > 1024) return (int)hipErrorInvalidValue;
  const int parts = nq <= 4 ? 64 : 256 / nq;               // a block for every CU
  hipLaunchKernelGGL(rank_kernel, dim3(parts, nq), dim3(1024), SORT_CAP * (sizeof(float) + sizeof(int)), stream, (const bf16*)corpus,
                     D, (const bf16*)queries, counts, cand, scores, cap, ks, kmax, out_ids, out_scores, out_count, host_count);
  const int rc = (int)hipGetLastError();
  return rc || host_count == nullptr ? rc : (int)hipStreamSynchronize(stream);
}
