// K13: Mixtral-style sparse MoE on CDNA4 fp8 MFMA (OCP e4m3; v_mfma_f32_16x16x32_fp8_fp8).
//
// Decode-step pipeline (every launch graph-capturable; buffers sized for the max batch):
//   1. moe_route:   router logits [T, E] -> softmax (f32), top-K, renormalise (HF Mixtral),
//                   counting sort of the T*K (token, expert) pairs by expert ->
//                   sorted token ids / routing weights, expert offsets [E+1], inverse map.
//   2. quant_rows:  dynamic per-row fp8 quantisation of the activations (scale = amax / 448).
//   3. moe_gemm<SILU>: per (expert, 32-row weight slice) workgroup: gathered token rows x W13_e
//                   (fp8 x fp8 MFMA, f32 acc), dequantised by row scales x weight scales, fused
//                   SiLU(gate) * up (16-row interleaved W13) -> [P, F] bf16.
//   4. quant_rows on [P, F], then moe_gemm<SCALE_W>: x W2_e, output scaled by the routing weight.
//   5. moe_combine: out[t] = sum over its K pairs (inverse map, no atomics).
// Weights are pre-tiled (ops/moe.py tile_fp8_weight): fragment pair (row group, 2 k-steps) is
// 1 KiB contiguous -- lane 16g+r holds 16 contiguous k of row r, feeding both MFMAs of the pair --
// so each weight load is one coalesced 16-byte-per-lane instruction, and the activation operand
// (same k permutation) is one 16-byte load per token row too; fp8 halves the bytes streamed per
// decode step versus bf16 (the whole expert bank is touched at decode batch sizes).
#include "common.h"

#define FP8_MAX 448.0f

// ---------------------------------------------------------------------------------------------
// 1. routing (single workgroup; T*K <= MOE_ROUTE_CAP pairs, E <= 64: decode batches)
// ---------------------------------------------------------------------------------------------
#define MOE_ROUTE_CAP 4096

__global__ void __launch_bounds__(1024) moe_route_kernel(const bf16* __restrict__ logits, int T, int E, int K,
                                                         int* __restrict__ sorted_tok, float* __restrict__ sorted_w,
                                                         int* __restrict__ offsets, int* __restrict__ inv) {
  __shared__ int cnt[64], cur[64];
  __shared__ int pe[MOE_ROUTE_CAP];    // expert of pair (t, j)
  __shared__ float pw[MOE_ROUTE_CAP];  // renormalised routing weight of pair (t, j)
  for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[e] = 0;
  __syncthreads();
  // pass 1: softmax (f32) + top-K + renormalise per token; count pairs per expert
  for (int t = threadIdx.x; t < T; t += blockDim.x) {
    float p[64];
    float mx = -INFINITY;
    for (int e = 0; e < E; ++e) {
      p[e] = (float)logits[(long)t * E + e];
      mx = fmaxf(mx, p[e]);
    }
    for (int e = 0; e < E; ++e) p[e] = __expf(p[e] - mx);
    float ws = 0.f;
    for (int j = 0; j < K; ++j) {
      int best = 0;
      for (int e = 1; e < E; ++e)
        if (p[e] > p[best]) best = e;
      atomicAdd(&cnt[best], 1);
      pe[t * K + j] = best;
      pw[t * K + j] = p[best];
      ws += p[best];
      p[best] = -1.f;
    }
    for (int j = 0; j < K; ++j) pw[t * K + j] /= ws;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int acc = 0;
    for (int e = 0; e < E; ++e) {
      offsets[e] = acc;
      cur[e] = acc;
      acc += cnt[e];
    }
    offsets[E] = acc;
  }
  __syncthreads();
  // pass 2: scatter pairs into their expert buckets (order inside a bucket is irrelevant: every
  // pair's rows are computed independently)
  for (int i = threadIdx.x; i < T * K; i += blockDim.x) {
    const int pos = atomicAdd(&cur[pe[i]], 1);
    inv[i] = pos;
    sorted_tok[pos] = i / K;
    sorted_w[pos] = pw[i];
  }
}

// ---------------------------------------------------------------------------------------------
// 1b. prefill routing + activation quantisation (any T): two launches instead of the torch
//     softmax / top-k / renormalise / argsort / bincount / cumsum / gather chain plus quant_rows.
//   moe_route_quant: one workgroup per token. Wave 0 routes it (one expert per lane: f32 softmax
//     numerators, K rounds of wave arg-max -- ties to the smaller expert id -- renormalised over the
//     top K, as moe_route_kernel); all four waves quantise the token's hidden row to e4m3 with the
//     row held in registers between the amax and the convert sweeps (read from HBM once).
//   moe_bucket: one workgroup counts the T*K pairs per expert in LDS, scans the offsets and
//     scatters the pairs into their buckets (order inside a bucket is irrelevant -- rows are
//     computed independently -- so the result is deterministic per row).
// ---------------------------------------------------------------------------------------------
// token t's experts by one wave, lane e holding logit e
__device__ __forceinline__ void moe_choose(float l, long t, int E, int K, int* __restrict__ pe, float* __restrict__ pw) {
  const int lane = threadIdx.x & 63;
  float mx = l;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  float p = lane < E ? __expf(l - mx) : -1.f;
  if (p != p) p = 0.f;                     // a total order: K experts are chosen whatever the logits
  float ws = 0.f, mine = 0.f;
  int myj = -1;
  for (int j = 0; j < K; ++j) {
    float bv = p;
    int bi = lane;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    ws += bv;
    if (lane == bi) { mine = p; myj = j; p = -1.f; }
  }
  if (myj >= 0) {
    pe[t * K + myj] = lane;
    pw[t * K + myj] = mine / ws;
  }
}

template <int CPT>
__global__ void __launch_bounds__(256) moe_route_quant_kernel(const bf16* __restrict__ x, int ldx, int H,
                                                              const bf16* __restrict__ logits, int E, int K,
                                                              unsigned char* __restrict__ q, float* __restrict__ scale,
                                                              int* __restrict__ pe, float* __restrict__ pw) {
  __shared__ float red[4];
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63;
  if (threadIdx.x < 64) moe_choose(lane < E ? (float)logits[t * E + lane] : -INFINITY, t, E, K, pe, pw);
  const uint4* xr = reinterpret_cast<const uint4*>(x + t * ldx);
  const int nchunk = H >> 3;
  float a[CPT][8];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = threadIdx.x + i * 256;
    if (c < nchunk) {
      unpack8(xr[c], a[i]);
#pragma unroll
      for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(a[i][k]));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
  if (lane == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float sc = amax > 0.f ? amax / FP8_MAX : 1.f;
  const float inv = 1.f / sc;
  if (threadIdx.x == 0) scale[t] = sc;
  uint2* qr = reinterpret_cast<uint2*>(q + t * (long)H);
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = threadIdx.x + i * 256;
    if (c < nchunk) {
      uint32_t w0 = 0, w1 = 0;
      w0 = __builtin_amdgcn_cvt_pk_fp8_f32(a[i][0] * inv, a[i][1] * inv, w0, false);
      w0 = __builtin_amdgcn_cvt_pk_fp8_f32(a[i][2] * inv, a[i][3] * inv, w0, true);
      w1 = __builtin_amdgcn_cvt_pk_fp8_f32(a[i][4] * inv, a[i][5] * inv, w1, false);
      w1 = __builtin_amdgcn_cvt_pk_fp8_f32(a[i][6] * inv, a[i][7] * inv, w1, true);
      qr[c] = make_uint2(w0, w1);
    }
  }
}

// pairs by their expert: counts, offsets and the scatter (order inside a bucket is irrelevant), by one block
__device__ __forceinline__ void moe_bucket(const int* __restrict__ pe, const float* __restrict__ pw, int P, int E, int K,
                                           int* __restrict__ sorted_tok, float* __restrict__ sorted_w,
                                           int* __restrict__ offsets, int* __restrict__ inv) {
  __shared__ int cnt[64], cur[64];
  for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[e] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < P; i += blockDim.x) atomicAdd(&cnt[pe[i]], 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    int acc = 0;
    for (int e = 0; e < E; ++e) {
      offsets[e] = acc;
      cur[e] = acc;
      acc += cnt[e];
    }
    offsets[E] = acc;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < P; i += blockDim.x) {
    const int pos = atomicAdd(&cur[pe[i]], 1);
    inv[i] = pos;
    sorted_tok[pos] = i / K;
    sorted_w[pos] = pw[i];
  }
}

__global__ void __launch_bounds__(1024) moe_bucket_kernel(const int* __restrict__ pe, const float* __restrict__ pw,
                                                          int P, int E, int K, int* __restrict__ sorted_tok,
                                                          float* __restrict__ sorted_w, int* __restrict__ offsets,
                                                          int* __restrict__ inv) {
  moe_bucket(pe, pw, P, E, K, sorted_tok, sorted_w, offsets, inv);
}

// ---------------------------------------------------------------------------------------------
// 2. dynamic per-row fp8 quantisation (one workgroup per row; row length multiple of 8)
// ---------------------------------------------------------------------------------------------
// The row stays in registers between the two sweeps, its CPT 16-byte pieces of a thread in one trip (96 rows of 14336: 4.8 us; read
// twice, a piece at a time, 7.1); a row of more than 8 pieces (16384 values) goes through the caches twice.
__device__ __forceinline__ uint2 fp8_of(const float (&f)[8], float inv) {
  uint32_t w0 = 0, w1 = 0;
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0] * inv, f[1] * inv, w0, false);
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2] * inv, f[3] * inv, w0, true);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[4] * inv, f[5] * inv, w1, false);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[6] * inv, f[7] * inv, w1, true);
  return make_uint2(w0, w1);
}
template <int CPT>
__global__ void __launch_bounds__(256) quant_rows_kernel(const bf16* __restrict__ x, int ld, int n, unsigned char* __restrict__ q,
                                                         float* __restrict__ scale) {
  constexpr bool HELD = CPT > 0;                             // 0: rows of any length
  __shared__ float red[4];
  const int row = blockIdx.x, chunks = n / 8;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (long)row * ld);
  uint4 v[HELD ? CPT : 1];
  float amax = 0.f;
  auto most = [&](const uint4& u) {
    float f[8];
    unpack8(u, f);
#pragma unroll
    for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(f[k]));
  };
  if constexpr (HELD) {
    if (chunks > 0) {                                        // behind the row's end its last piece again
#pragma unroll
      for (int i = 0; i < CPT; ++i) v[i] = xr[min((int)threadIdx.x + 256 * i, chunks - 1)];
#pragma unroll
      for (int i = 0; i < CPT; ++i) most(v[i]);
    }
  } else {
    for (int c = threadIdx.x; c < chunks; c += 256) most(xr[c]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = amax > 0.f ? amax / FP8_MAX : 1.f;
  const float inv = 1.f / s;
  if (threadIdx.x == 0) scale[row] = s;
  uint2* qr = reinterpret_cast<uint2*>(q + (long)row * n);
  auto put = [&](const uint4& u, int c) {
    float f[8];
    unpack8(u, f);
    qr[c] = fp8_of(f, inv);
  };
  if constexpr (HELD) {
#pragma unroll
    for (int i = 0; i < CPT; ++i)
      if ((int)threadIdx.x + 256 * i < chunks) put(v[i], threadIdx.x + 256 * i);
  } else {
    for (int c = threadIdx.x; c < chunks; c += 256) put(xr[c], c);
  }
}

// 2a. decode batches: router, choice, quantised row and buckets in one launch, a block per token.  Every block reads the router
//     (8 experts of 4096: 64 KB) from the caches; logits are f32 sums rounded to bf16, as a bf16 product's.  The block that draws the
//     last ticket sorts the pairs into their buckets.  48 tokens: 9 us, for the library's product (13.4), moe_route_kernel (9) and
//     quant_rows_kernel (4.6); ops/moe.py has the number of tokens from which those three are the shorter way.
template <int CPT, int EM>
__global__ void __launch_bounds__(256) moe_decode_route_kernel(const bf16* __restrict__ x, int ldx, int H, const bf16* __restrict__ rw,
                                                               int T, int E, int K, unsigned char* __restrict__ q,
                                                               float* __restrict__ scale, int* pe, float* pw, int* ticket,
                                                               int* __restrict__ sorted_tok, float* __restrict__ sorted_w,
                                                               int* __restrict__ offsets, int* __restrict__ inv_pos) {
  __shared__ float red[4], part[4][EM];
  __shared__ int last;
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, chunks = H / 8;
  const uint4* xr = reinterpret_cast<const uint4*>(x + t * ldx);
  uint4 v[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = threadIdx.x + 256 * i;
    v[i] = c < chunks ? xr[c] : uint4{0, 0, 0, 0};
  }
  float amax = 0.f, sum[EM];
#pragma unroll
  for (int e = 0; e < EM; ++e) sum[e] = 0.f;
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = min((int)threadIdx.x + 256 * i, chunks - 1);
    uint4 r[EM];
#pragma unroll
    for (int e = 0; e < EM; ++e) r[e] = reinterpret_cast<const uint4*>(rw + (long)min(e, E - 1) * H)[c];
    float f[8];
    unpack8(v[i], f);
#pragma unroll
    for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(f[k]));
    if ((int)threadIdx.x + 256 * i >= chunks) continue;      // (not 0 x a weight, which may be infinite)
#pragma unroll
    for (int e = 0; e < EM; ++e) {
      float g[8];
      unpack8(r[e], g);
#pragma unroll
      for (int k = 0; k < 8; ++k) sum[e] += f[k] * g[k];
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
#pragma unroll
  for (int e = 0; e < EM; ++e) sum[e] = wave_sum(sum[e]);
  if (lane == 0) {
    red[w] = amax;
#pragma unroll
    for (int e = 0; e < EM; ++e) part[w][e] = sum[e];
  }
  __syncthreads();
  if (w == 0) {
    const int e = min(lane, EM - 1);
    const float l = (float)(bf16)((part[0][e] + part[1][e]) + (part[2][e] + part[3][e]));
    moe_choose(lane < E ? l : -INFINITY, t, E, K, pe, pw);
  }
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = amax > 0.f ? amax / FP8_MAX : 1.f;
  const float inv = 1.f / s;
  if (threadIdx.x == 0) scale[t] = s;
  uint2* qr = reinterpret_cast<uint2*>(q + t * (long)H);
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c >= chunks) continue;
    float f[8];
    unpack8(v[i], f);
    qr[c] = fp8_of(f, inv);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (threadIdx.x == 0) {                                    // of the wave that stored the pairs
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == T - 1;
    if (last) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      *ticket = 0;                                           // for the next launch
    }
  }
  __syncthreads();
  if (last) moe_bucket(pe, pw, T * K, E, K, sorted_tok, sorted_w, offsets, inv_pos);
}

// 2b. prefill experts: SiLU(gate) * up of the 16-row-interleaved W13 GEMM output, quantised per row
//     to fp8 in the same pass (one workgroup per row, the row held in registers between the amax
//     and the quantise sweeps): the bf16 activation never round-trips through HBM.
template <int CPT>
__global__ void __launch_bounds__(256) silu_quant_rows_kernel(const bf16* __restrict__ gu, int F,
                                                              unsigned char* __restrict__ q,
                                                              float* __restrict__ scale) {
  __shared__ float red[4];
  const long row = blockIdx.x;
  const uint4* gr = reinterpret_cast<const uint4*>(gu + row * 2L * F);
  const int nchunk = F >> 3;   // 8 outputs per chunk: output cols 8c..8c+7 = pair c/2, half c&1
  float a[CPT][8];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = threadIdx.x + i * 256;
    if (c < nchunk) {
      float g[8], u[8];
      const int pair = c >> 1, half = c & 1;
      unpack8(gr[pair * 4 + half], g);
      unpack8(gr[pair * 4 + 2 + half], u);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        // silu in the activation dtype, like silu_mul_kernel: bf16(silu(g)) * u, rounded to bf16
        a[i][k] = (float)(bf16)((float)(bf16)(g[k] / (1.f + __expf(-g[k]))) * u[k]);
        amax = fmaxf(amax, fabsf(a[i][k]));
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float sc = amax > 0.f ? amax / FP8_MAX : 1.f;
  const float inv = 1.f / sc;
  if (threadIdx.x == 0) scale[row] = sc;
  uint2* qr = reinterpret_cast<uint2*>(q + row * (long)F);
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = threadIdx.x + i * 256;
    if (c < nchunk) {
      uint32_t w0 = 0, w1 = 0;
      w0 = __builtin_amdgcn_cvt_pk_fp8_f32(a[i][0] * inv, a[i][1] * inv, w0, false);
      w0 = __builtin_amdgcn_cvt_pk_fp8_f32(a[i][2] * inv, a[i][3] * inv, w0, true);
      w1 = __builtin_amdgcn_cvt_pk_fp8_f32(a[i][4] * inv, a[i][5] * inv, w1, false);
      w1 = __builtin_amdgcn_cvt_pk_fp8_f32(a[i][6] * inv, a[i][7] * inv, w1, true);
      qr[c] = make_uint2(w0, w1);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// 3/4. grouped fp8 GEMM over expert buckets
// ---------------------------------------------------------------------------------------------
#define MOE_EPI_SILU 1
#define MOE_EPI_ROUTEW 2

// One chunk of up to 16 * MT pairs (c0 ..) of expert e against the workgroup's 16 * NTF weight rows.  The weights are streamed once and
// bound the kernel, so what counts is how they stream: D k-pairs of weights and activations are asked for ahead of the MFMAs, past the
// caches' replacement (ONCE), and only the MT token tiles that hold pairs are read and multiplied.  8 experts of 2 x 14336 x 4096, 48
// tokens: first product 182 -> 145 us (6.4 TB/s; 138, 6.8, for 16 tokens), second 87 -> 72; one k-pair ahead, four token tiles whatever
// the rows and 64 KB of LDS a workgroup before.  Without ONCE 152 and 80; four pairs or six ahead the same; four workgroups a CU
// instead of three 197 and 100.
template <int NTF, int NW, int EPI, int MT, int D, bool ONCE = true>
__device__ __forceinline__ void moe_chunk(const unsigned char* __restrict__ Xq, const float* __restrict__ xs, const int* __restrict__ rows,
                                          const unsigned char* __restrict__ We, const float* __restrict__ wse,
                                          const float* __restrict__ route_w, bf16* __restrict__ Y, int N, int K, int n0, int c0, int nrow,
                                          float* red) {
  constexpr int NR = 16 * NTF, RS = 20;                       // RS: a row's 16 sums; 4 rows on, the banks behind them
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, col = lane & 15;
  const int kper = K / NW, kb = w * kper, kp = kper / 64;
  const long kpairs = K / 64;
  // lane (g, col) owns physical k = 64p + 16g .. +15 of its token row: one 16-B load per row tile
  // and k-pair, matching the weight tiling (ops/moe.py tile_fp8_weight); bytes 0-7 feed the
  // first MFMA of the pair, bytes 8-15 the second
  const unsigned char* xr[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int pr = c0 + min(16 * m + col, nrow - 1);
    xr[m] = Xq + (long)(rows ? rows[pr] : pr) * K + kb + 16 * g;
  }
  const unsigned char* wr = We + ((n0 / 16 * kpairs + kb / 64) * 64 + lane) * 16;
  f32x4 acc[NTF][MT];
#pragma unroll
  for (int f = 0; f < NTF; ++f)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[f][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
  u32x4_t wv[D][NTF], xv[D][MT];
  auto fetch = [&](int slot, int p) {
#pragma unroll
    for (int f = 0; f < NTF; ++f) {
      const u32x4_t* src = reinterpret_cast<const u32x4_t*>(wr + (f * kpairs + p) * 1024);
      wv[slot][f] = ONCE ? __builtin_nontemporal_load(src) : *src;
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) xv[slot][m] = *reinterpret_cast<const u32x4_t*>(xr[m] + 64 * p);
  };
  auto use = [&](int slot) {
    // both k-halves of one accumulator back to back (a dependent MFMA pair): interleaving the
    // halves across all accumulators made hipcc shuffle them between AGPRs every pair
#pragma unroll
    for (int f = 0; f < NTF; ++f) {
      const long a0 = ((long)wv[slot][f].y << 32 | wv[slot][f].x), a1 = ((long)wv[slot][f].w << 32 | wv[slot][f].z);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const long b0 = ((long)xv[slot][m].y << 32 | xv[slot][m].x), b1 = ((long)xv[slot][m].w << 32 | xv[slot][m].z);
        acc[f][m] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a0, b0, acc[f][m], 0, 0, 0);
        acc[f][m] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a1, b1, acc[f][m], 0, 0, 0);
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < kp) fetch(d, d);
  int p = 0;
  for (; p + 2 * D <= kp; p += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      use(d);
      fetch(d, p + D + d);
      if (MT == 1) __builtin_amdgcn_sched_barrier(0);
    }
  }
  for (; p < kp; p += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (p + d < kp) use(d);
      if (p + D + d < kp) fetch(d, p + D + d);
    }
  }
  // the waves' sums of K, one token tile at a time; a thread has two neighbouring outputs of a pair
  constexpr int OUTN = (EPI == MOE_EPI_SILU) ? NR / 2 : NR;
  const int ldy = (EPI == MOE_EPI_SILU) ? N / 2 : N;
  for (int m = 0; m < MT; ++m) {
    if (16 * m >= nrow) break;
    __syncthreads();                                          // the tile before has been read
    float* mine = red + w * NR * RS;
#pragma unroll
    for (int mm = 0; mm < MT; ++mm)
      if (mm == m)
#pragma unroll
        for (int f = 0; f < NTF; ++f)
#pragma unroll
          for (int r = 0; r < 4; ++r) mine[(16 * f + 4 * g + r) * RS + col] = acc[f][mm][r];
    __syncthreads();
    for (int idx = threadIdx.x; idx < 16 * (OUTN / 2); idx += NW * 64) {
      const int mr = idx / (OUTN / 2), c = idx % (OUTN / 2) * 2;
      if (16 * m + mr >= nrow) continue;
      const int pr = c0 + 16 * m + mr;
      const float sx = xs[rows ? rows[pr] : pr];
      bf16 o[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (EPI == MOE_EPI_SILU) {
          const int rg = 32 * (c >> 4) + (c & 15) + j, ru = rg + 16;
          float gs = 0.f, us = 0.f;
#pragma unroll
          for (int ww = 0; ww < NW; ++ww) {
            gs += red[(ww * NR + rg) * RS + mr];
            us += red[(ww * NR + ru) * RS + mr];
          }
          const float gv = (float)(bf16)(gs * sx * wse[n0 + rg]);
          const float uv = (float)(bf16)(us * sx * wse[n0 + ru]);
          o[j] = (bf16)((float)(bf16)(gv / (1.f + __expf(-gv))) * uv);
        } else {
          float s = 0.f;
#pragma unroll
          for (int ww = 0; ww < NW; ++ww) s += red[(ww * NR + c + j) * RS + mr];
          o[j] = (bf16)(s * sx * wse[n0 + c + j] * route_w[pr]);
        }
      }
      const int ncol = (EPI == MOE_EPI_SILU) ? n0 / 2 + c : n0 + c;
      *reinterpret_cast<uint32_t*>(Y + (long)pr * ldy + ncol) = *reinterpret_cast<const uint32_t*>(o);
    }
  }
}

// (two waves a SIMD asked for: left to itself the compiler packs the wide workgroup's registers for three, 128 tokens 198 us instead of 175)
template <int NTF, int NW, int EPI>
__global__ void __launch_bounds__(NW * 64, NTF == 4 ? 2 : 1) moe_gemm_kernel(
    const unsigned char* __restrict__ Xq, const float* __restrict__ xs, const int* __restrict__ rows,
    const int* __restrict__ offsets, const unsigned char* __restrict__ Wt, const float* __restrict__ ws,
    const float* __restrict__ route_w, bf16* __restrict__ Y, int N, int K) {
  __shared__ float red[NW * 16 * NTF * 20];
  const int e = blockIdx.y;
  const int p0 = offsets[e], p1 = offsets[e + 1];
  if (p1 <= p0) return;
  const int n0 = blockIdx.x * 16 * NTF;
  const unsigned char* We = Wt + (long)e * N * K;
  for (int c0 = p0; c0 < p1; c0 += 64) {  // token chunks of 64 pairs
    const int nrow = min(64, p1 - c0);
#define CHUNK(...) moe_chunk<NTF, NW, EPI, __VA_ARGS__>(Xq, xs, rows, We, ws + (long)e * N, route_w, Y, N, K, n0, c0, nrow, red)
    if (nrow <= 16) CHUNK(1, 4);
    else if (nrow <= 32) CHUNK(2, 3);
    else if (p1 - p0 <= 64) CHUNK(4, 2);
    else CHUNK(4, 2, false);   // (the next chunk reads the weights again)
#undef CHUNK
  }
}

// ---------------------------------------------------------------------------------------------
// 5. combine the K expert outputs of each token
// ---------------------------------------------------------------------------------------------
// W (optional, prefill path): routing weight of each sorted pair, applied here in f32 (the decode
// path already scaled its rows inside the W2 GEMM epilogue)
__global__ void moe_combine_kernel(const bf16* __restrict__ Y2, const int* __restrict__ inv,
                                   const float* __restrict__ W, int K, int H, bf16* __restrict__ out) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x; c < H / 8; c += blockDim.x) {
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int j = 0; j < K; ++j) {
      const int pos = inv[t * K + j];
      const float wj = W ? W[pos] : 1.f;
      float f[8];
      unpack8(reinterpret_cast<const uint4*>(Y2 + (long)pos * H)[c], f);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] += wj * f[i];
    }
    reinterpret_cast<uint4*>(out + (long)t * H)[c] = pack8(acc);
  }
}

PENNY_API int penny_moe_route(const void* logits, int T, int E, int K, int* sorted_tok, float* sorted_w, int* offsets,
                              int* inv, hipStream_t stream) {
  if (T <= 0) return 0;
  if (E > 64 || K > 8 || K > E || T * K > MOE_ROUTE_CAP) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(1024), 0, stream, (const bf16*)logits, T, E, K, sorted_tok,
                     sorted_w, offsets, inv);
  PENNY_RETURN_LAUNCH();
}

// prefill routing + quantisation: x [T, H] (row stride ldx) bf16, logits [T, E] bf16 ->
// xq [T, H] e4m3, xs [T]; pair expert / weight scratch pe, pw [T*K]; buckets sorted_tok /
// sorted_w [T*K], offsets [E+1], inverse map inv [T*K] (pair t*K+j -> sorted position)
PENNY_API int penny_moe_route_quant(const void* x, int ldx, const void* logits, int T, int H, int E, int K, void* xq,
                                    float* xs, int* pe, float* pw, int* sorted_tok, float* sorted_w, int* offsets,
                                    int* inv, hipStream_t stream) {
  if (T <= 0) return 0;
  if (E > 64 || K < 1 || K > 8 || K > E || H % 8 || ldx % 8) return (int)hipErrorInvalidValue;
  const int cpt = (H / 8 + 255) / 256;
#define RQ_CASE(C)                                                                                        \
  if (cpt <= C) {                                                                                         \
    hipLaunchKernelGGL(moe_route_quant_kernel<C>, dim3(T), dim3(256), 0, stream, (const bf16*)x, ldx, H, \
                       (const bf16*)logits, E, K, (unsigned char*)xq, xs, pe, pw);                       \
  } else
  RQ_CASE(1) RQ_CASE(2) RQ_CASE(4) RQ_CASE(8) return (int)hipErrorInvalidValue;
#undef RQ_CASE
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return (int)err;
  hipLaunchKernelGGL(moe_bucket_kernel, dim3(1), dim3(1024), 0, stream, pe, pw, T * K, E, K, sorted_tok, sorted_w,
                     offsets, inv);
  PENNY_RETURN_LAUNCH();
}

// penny_moe_route_quant for decode batches from the router's weight rw [E, H] bf16 in one launch: E <= 16, T K <= 4096, H / 8 <= 2048,
// 16-byte rows.  ticket: one int, zero at the first call, zero again behind every call.
PENNY_API int penny_moe_decode_route(const void* x, int ldx, const void* rw, int T, int H, int E, int K, void* xq, float* xs, int* pe,
                                     float* pw, int* ticket, int* sorted_tok, float* sorted_w, int* offsets, int* inv,
                                     hipStream_t stream) {
  if (T <= 0) return 0;
  if (E < 1 || E > 16 || K < 1 || K > 8 || K > E || (long)T * K > MOE_ROUTE_CAP || H < 8 || H % 8 || H > 16384 || ldx % 8 ||
      ((size_t)x | (size_t)rw) % 16)
    return (int)hipErrorInvalidValue;
  const int cpt = (H / 8 + 255) / 256;
#define ROUTE(C, EM)                                                                                                             \
  moe_decode_route_kernel<C, EM><<<T, 256, 0, stream>>>((const bf16*)x, ldx, H, (const bf16*)rw, T, E, K, (unsigned char*)xq, xs, \
                                                        pe, pw, ticket, sorted_tok, sorted_w, offsets, inv)
#define ROUTE_E(C)                \
  do {                            \
    if (E <= 8) ROUTE(C, 8);      \
    else ROUTE(C, 16);            \
  } while (0)
  if (cpt <= 1) ROUTE_E(1);
  else if (cpt <= 2) ROUTE_E(2);
  else if (cpt <= 4) ROUTE_E(4);
  else ROUTE_E(8);
#undef ROUTE_E
#undef ROUTE
  PENNY_RETURN_LAUNCH();
}

// gu [rows, 2F] bf16 (16-column-interleaved gate|up) -> q [rows, F] e4m3, scale [rows] f32
PENNY_API int penny_silu_quant_rows_fp8(const void* gu, int rows, int F, void* q, float* scale, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (F % 16) return (int)hipErrorInvalidValue;
  const int cpt = (F / 8 + 255) / 256;
#define SQ_CASE(C)                                                                                        \
  if (cpt <= C) {                                                                                         \
    hipLaunchKernelGGL(silu_quant_rows_kernel<C>, dim3(rows), dim3(256), 0, stream, (const bf16*)gu, F,   \
                       (unsigned char*)q, scale);                                                         \
    PENNY_RETURN_LAUNCH();                                                                                \
  }
  SQ_CASE(1) SQ_CASE(2) SQ_CASE(4) SQ_CASE(8) SQ_CASE(16)
#undef SQ_CASE
  return (int)hipErrorInvalidValue;
}

PENNY_API int penny_quant_rows_fp8(const void* x, int ld, int rows, int n, void* q, float* scale, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (n % 8) return (int)hipErrorInvalidValue;
  const int cpt = (n / 8 + 255) / 256;
#define QUANT(C) quant_rows_kernel<C><<<rows, 256, 0, stream>>>((const bf16*)x, ld, n, (unsigned char*)q, scale)
  if (cpt <= 1) QUANT(1);
  else if (cpt <= 2) QUANT(2);
  else if (cpt <= 4) QUANT(4);
  else if (cpt <= 8) QUANT(8);
  else QUANT(0);
#undef QUANT
  PENNY_RETURN_LAUNCH();
}

template <int NTF>
static int moe_gemm_launch(const void* Xq, const float* xs, const int* rows, const int* offsets, const void* Wt,
                           const float* ws, const float* route_w, void* Y, int E, int N, int K, int epi,
                           hipStream_t stream) {
  dim3 grid(N / (16 * NTF), E);
  // Waves split K into whole 64-wide k-pairs.  Thin workgroups (NTF 2) want long streams a wave: 2 waves up to K = 8192 (4096, 48 / 64 / 96
  // tokens: 143 / 154 / 180 us, 4 waves 146 / 162 / 190), 8 beyond, where they are taken because few of them fill the chip (14336, one
  // token 18.7, 4 waves 24.7).  NTF 4: 4 waves (4096, 128 tokens 175, 2 waves 184).
#define MOE_LAUNCH(NW_)                                                                                          \
  {                                                                                                              \
    if (epi == MOE_EPI_SILU)                                                                                     \
      hipLaunchKernelGGL((moe_gemm_kernel<NTF, NW_, MOE_EPI_SILU>), grid, dim3(NW_ * 64), 0, stream,            \
                         (const unsigned char*)Xq, xs, rows, offsets, (const unsigned char*)Wt, ws, route_w,     \
                         (bf16*)Y, N, K);                                                                        \
    else                                                                                                         \
      hipLaunchKernelGGL((moe_gemm_kernel<NTF, NW_, MOE_EPI_ROUTEW>), grid, dim3(NW_ * 64), 0, stream,          \
                         (const unsigned char*)Xq, xs, rows, offsets, (const unsigned char*)Wt, ws, route_w,     \
                         (bf16*)Y, N, K);                                                                        \
  }
  if (NTF == 2 && K % 128 == 0 && K < 8192) MOE_LAUNCH(2)
  else if (NTF == 2 && K % 512 == 0) MOE_LAUNCH(8)
  else if (K % 256 == 0) MOE_LAUNCH(4)
  else if (K % 128 == 0) MOE_LAUNCH(2)
  else MOE_LAUNCH(1)
#undef MOE_LAUNCH
  PENNY_RETURN_LAUNCH();
}

// epi 1: SiLU-gated (W13 interleaved, Y [P, N/2]); epi 2: scale by routing weight (Y [P, N]).
// ntf: 16-row weight groups per workgroup (2 or 4).
PENNY_API int penny_moe_gemm_fp8(const void* Xq, const float* xs, const int* rows, const int* offsets, const void* Wt,
                                 const float* ws, const float* route_w, void* Y, int E, int N, int K, int epi,
                                 int ntf, hipStream_t stream) {
  if ((ntf != 2 && ntf != 4) || N % (16 * ntf) || K % 64) return (int)hipErrorInvalidValue;
  if (ntf == 4) return moe_gemm_launch<4>(Xq, xs, rows, offsets, Wt, ws, route_w, Y, E, N, K, epi, stream);
  return moe_gemm_launch<2>(Xq, xs, rows, offsets, Wt, ws, route_w, Y, E, N, K, epi, stream);
}

PENNY_API int penny_moe_combine(const void* Y2, const int* inv, int T, int K, int H, void* out, hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T), dim3(256), 0, stream, (const bf16*)Y2, inv, (const float*)nullptr,
                     K, H, (bf16*)out);
  PENNY_RETURN_LAUNCH();
}

// out[t] = sum_j W[inv[t*K+j]] * Y2[inv[t*K+j]]  (f32 accumulate; prefill combine, no atomics)
PENNY_API int penny_moe_combine_weighted(const void* Y2, const int* inv, const float* W, int T, int K, int H,
                                         void* out, hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T), dim3(256), 0, stream, (const bf16*)Y2, inv, W, K, H, (bf16*)out);
  PENNY_RETURN_LAUNCH();
}
