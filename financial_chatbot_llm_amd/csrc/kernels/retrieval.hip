// K15: filtered exact top-k similarity search over an HBM-resident corpus (replaces Qdrant's
// filtered HNSW query, tools/qdrant_tool.py:98-153).
//
// Filters are the reference's: user_id == u (always) AND date >= t (optional).  Such filters are
// very selective (one user's rows out of ~1M), so the search is organised around the filter, not
// the vectors:
//   1. filter_compact: one pass over the int32 user codes (and, near a match, the int64 dates)
//      evaluates every query's filter and appends matching row ids to a per-query
//      candidate list (wave-aggregated atomics).  Vectors of non-matching rows are never read.
//   2. score: one wave per candidate row computes <corpus_row, query> (768-d bf16, 16 B/lane).
//   3. select: one workgroup per query ranks up to SORT_CAP (score, row) pairs in LDS,
//      descending by score, ties by row id, and writes the first k.
// Queries with more candidates than SORT_CAP are finished by the caller (torch.topk on the
// device-side score list), which the host detects from the returned counts.
#include "common.h"

#define SORT_CAP 8192
#define CSTRIDE 32      // counters lie a cache line apart: beside each other, their atomics wait for one another

// A block takes FROWS * 256 rows at a time, a thread FROWS of them, 256 apart; the codes and the queries are fetched together.
// Dates are read only where a row of the wave belongs to a queried user.  Bound by latency and the code comparisons (1M rows,
// 16 queries: 11 us; one row per thread, dates always read, counters side by side, 14).
constexpr int FROWS = 4;
__global__ void __launch_bounds__(256) filter_compact_kernel(const int* __restrict__ user_codes,
                                                             const long long* __restrict__ dates, long N,
                                                             const int* __restrict__ q_user,
                                                             const long long* __restrict__ q_floor, int nq,
                                                             int* __restrict__ counts, int* __restrict__ cand, int cap) {
  __shared__ int su[64];
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
      if (threadIdx.x < nq) {
        su[threadIdx.x] = q_user[threadIdx.x];
        sf[threadIdx.x] = q_floor[threadIdx.x];
      }
      __syncthreads();
      first = false;
    }
    bool any = false;
    for (int qi = 0; qi < nq; ++qi) {
      const int u = su[qi];
#pragma unroll
      for (int r = 0; r < FROWS; ++r) any |= code[r] == u;
    }
    if (!__any(any)) continue;
    long long d[FROWS];
#pragma unroll
    for (int r = 0; r < FROWS; ++r) d[r] = dates[in[r] ? base + 256 * r + threadIdx.x : N - 1];
    for (int qi = 0; qi < nq; ++qi) {
      unsigned long long mask[FROWS];
      int hits = 0;
#pragma unroll
      for (int r = 0; r < FROWS; ++r) {
        mask[r] = __ballot(in[r] && code[r] == su[qi] && d[r] >= sf[qi]);
        hits += __popcll(mask[r]);
      }
      if (hits == 0) continue;
      int start = 0;
      if (lane == 0) start = atomicAdd(&counts[qi * CSTRIDE], hits);
      start = __shfl(start, 0, 64);
#pragma unroll
      for (int r = 0; r < FROWS; ++r) {
        const int pos = start + __popcll(mask[r] & ((1ull << lane) - 1ull));
        if ((mask[r] >> lane & 1) && pos < cap) cand[(long)qi * cap + pos] = (int)(base + 256 * r + threadIdx.x);
        start += __popcll(mask[r]);
      }
    }
  }
}

// one wave per (query, candidate); D multiple of 8, D <= 1024
__global__ void score_kernel(const bf16* __restrict__ corpus, int D, const bf16* __restrict__ queries,
                             const int* __restrict__ counts, const int* __restrict__ cand, int cap,
                             float* __restrict__ scores) {
  const int qi = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int waves = (gridDim.x * blockDim.x) >> 6;
  const int wid = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int cnt = min(counts[qi * CSTRIDE], cap);
  const int nch = D >> 3;
  float qv[2][8];
  for (int r = 0; r < 2; ++r) {
    const int c = lane + 64 * r;
    if (c < nch) unpack8(reinterpret_cast<const uint4*>(queries + (long)qi * D)[c], qv[r]);
  }
  for (int i = wid; i < cnt; i += waves) {
    const int row = cand[(long)qi * cap + i];
    const uint4* cr = reinterpret_cast<const uint4*>(corpus + (long)row * D);
    float acc = 0.f;
    for (int r = 0; r < 2; ++r) {
      const int c = lane + 64 * r;
      if (c < nch) {
        float f[8];
        unpack8(cr[c], f);
#pragma unroll
        for (int k = 0; k < 8; ++k) acc += f[k] * qv[r][k];
      }
    }
    acc = wave_sum(acc);
    if (lane == 0) scores[(long)qi * cap + i] = acc;
  }
}

__device__ __forceinline__ bool before(float sa, int ia, float sb, int ib) {  // a ranks before b
  return sa > sb || (sa == sb && ia < ib);
}

// One block per query: the first k of its candidates, -1 / 0 behind them, the count to the device and (host_count) to the host,
// and counts back to zero for the next call.  Up to RANK_CAP candidates each finds its rank by counting those before it, 1024
// threads over all pairs (16 queries of about 90: 5 us; the sort's 28 barriers took 10); more are sorted.
constexpr int RANK_CAP = 256;
__global__ void __launch_bounds__(1024) select_kernel(int* __restrict__ counts, const int* __restrict__ cand,
                                                      const float* __restrict__ scores, int cap,
                                                      const int* __restrict__ ks, int kmax, int* __restrict__ out_ids,
                                                      float* __restrict__ out_scores, int* __restrict__ out_count,
                                                      int* __restrict__ host_count) {
  extern __shared__ __attribute__((aligned(16))) char dyn[];
  float* ss = reinterpret_cast<float*>(dyn);
  int* si = reinterpret_cast<int*>(dyn + SORT_CAP * sizeof(float));
  __shared__ int rank[RANK_CAP];
  const int qi = blockIdx.x;
  const int total = counts[qi * CSTRIDE];
  const int cnt = min(total, cap);
  const bool big = total > SORT_CAP;                       // the host finishes this query
  const int k = big ? 0 : min(ks[qi], min(cnt, kmax));
  for (int i = max(k, 0) + threadIdx.x; i < kmax; i += blockDim.x) {
    out_ids[(long)qi * kmax + i] = -1;
    out_scores[(long)qi * kmax + i] = 0.f;
  }
  if (threadIdx.x == 0) {
    out_count[qi] = big ? -total : k;
    if (host_count != nullptr) host_count[qi] = big ? -total : k;
  }
  if (big || cnt == 0) {
    __syncthreads();                                       // everybody has read the count
    if (threadIdx.x == 0) counts[qi * CSTRIDE] = 0;
    return;
  }
  int n = 1;
  while (n < cnt) n <<= 1;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const bool v = i < cnt;
    ss[i] = v ? scores[(long)qi * cap + i] : -INFINITY;
    si[i] = v ? cand[(long)qi * cap + i] : 0x7fffffff;
    if (i < RANK_CAP) rank[i] = 0;
  }
  __syncthreads();
  if (threadIdx.x == 0) counts[qi * CSTRIDE] = 0;
  if (cnt <= RANK_CAP) {
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
    return;
  }
  for (int size = 2; size <= n; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int j = i ^ stride;
        if (j > i) {
          const bool desc = (i & size) == 0;  // this run sorted "best first"
          const bool swap = desc ? before(ss[j], si[j], ss[i], si[i]) : before(ss[i], si[i], ss[j], si[j]);
          if (swap) {
            const float t = ss[i]; ss[i] = ss[j]; ss[j] = t;
            const int u = si[i]; si[i] = si[j]; si[j] = u;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < k; i += blockDim.x) {
    out_ids[(long)qi * kmax + i] = si[i];
    out_scores[(long)qi * kmax + i] = ss[i];
  }
}

// counts [nq][32]: zero at the first call, zero again behind every call.  host_count (pinned host memory, or null): out_count as
// well, there once the stream has been waited for.
PENNY_API int penny_filtered_topk(const void* corpus, const int* user_codes, const long long* dates, long N, int D,
                                  const void* queries, const int* q_user, const long long* q_floor, const int* ks,
                                  int nq, int kmax, int* counts, int* cand, float* scores, int cap, int* out_ids,
                                  float* out_scores, int* out_count, int* host_count, hipStream_t stream) {
  if (nq <= 0) return 0;
  if (nq > 64 || D % 8 || D > 1024) return (int)hipErrorInvalidValue;
  long g = (N + 256 * FROWS - 1) / (256 * FROWS);
  if (g > 4096) g = 4096;
  if (g < 1) g = 1;
  hipLaunchKernelGGL(filter_compact_kernel, dim3((int)g), dim3(256), 0, stream, user_codes, dates, N, q_user, q_floor,
                     nq, counts, cand, cap);
  hipLaunchKernelGGL(score_kernel, dim3(64, nq), dim3(256), 0, stream, (const bf16*)corpus, D, (const bf16*)queries,
                     counts, cand, cap, scores);
  const size_t lds = SORT_CAP * (sizeof(float) + sizeof(int));
  hipLaunchKernelGGL(select_kernel, dim3(nq), dim3(1024), lds, stream, counts, cand, scores, cap, ks, kmax, out_ids,
                     out_scores, out_count, host_count);
  PENNY_RETURN_LAUNCH();
}
