// BERT / bge encoder (K14) kernels of their own: bidirectional attention straight over the packed QKV rows, and the
// biased projections of small batches.
//
//   penny_encoder_attention   every text attends within itself; most are short (a query or a transaction: 6 - 128
//                             tokens), so a 64-token tile of one (text, head) is about a whole problem, and no paged cache
//                             is written first.
//   penny_gemm_bias_small     bf16(x w^T + b) [-> exact GELU] for up to some two thousand rows, most of them on gemm_splitk.hip's tiles.
//   penny_encoder_embed       word + position + type rows and their layer norm in one pass.
//   penny_encoder_layers      the launches of all layers of a small batch, from one call.
//   penny_encoder_pool        the texts' first rows, normalised.
#include "common.h"

namespace {

union Frag {
  uint4 u;
  bf16x8 v;
};

typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// grid (query tiles of 64, heads, texts), 4 waves of 16 queries.  qkv [T, ld]: q | k | v, heads side by side.  Per tile of
// 64 keys: keys and values to LDS as they lie, each row once, the rows behind the text's end not at all; S^T = K Q^T, online softmax
// in base 2, O^T += V^T P^T with the values through the transposing LDS read and P straight from the score registers (K slot 8 g + i
// holds keys 4 g + i and 16 + 4 g + i); sixteens of keys behind the end are left out.  LDS rows are 16 bytes longer than their values, so
// that 16 of them start in different banks.  Bound by the QKV rows read and the output written: 1024 texts of 6 - 64 tokens
// (36k), 12 heads of 64: 40 us (5.6 TB/s); with each wave reading the keys for itself, outputs in 8-byte pieces and the values transposed on
// the way in 59; the paged form took 202 us for the cache write and 72 us for the attention.
// Longer texts read each other's keys once per 64 queries, without prefetch (32,768 tokens, us, that form / this / paged write + attention:
// texts of 128 72 / 47 / 239 + 39, of 512 224 / 160 / 237 + 100; 8 texts of 512 36 / 29 / 25 + 20).
template <int D>
__global__ void __launch_bounds__(256) encoder_attention_kernel(const bf16* __restrict__ qkv, long ld,
                                                                const int* __restrict__ cu, int H, float scale_log2,
                                                                bf16* __restrict__ out) {
  constexpr int KS = D / 32, NT = D / 16, CP = D / 8, RB = D + 8, LN = 64 * CP / 256;
  __shared__ __attribute__((aligned(16))) bf16 kt[64 * RB], vt[64 * RB];
  const int r0 = cu[blockIdx.z], n = cu[blockIdx.z + 1] - r0, t0 = blockIdx.x * 64;
  if (t0 >= n) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15, h = blockIdx.y;
  const bf16* q = qkv + (long)r0 * ld + h * D;
  const bf16* k = q + H * D;
  const bf16* v = k + H * D;
  const int qi = t0 + 16 * w + c;
  const bool live = t0 + 16 * w < n;                 // this wave has a query
  Frag qf[KS];
  if (live) {
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s].u = *reinterpret_cast<const uint4*>(q + min(qi, n - 1) * ld + 32 * s + 8 * g);
  }
  f32x4 o[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  for (int k0 = 0; k0 < n; k0 += 64) {
    uint4 kk[LN], vv[LN];
#pragma unroll
    for (int i = 0; i < LN; ++i) {                   // a thread's 16 bytes of a key and a value, zeros behind the text's end
      const int e = threadIdx.x + 256 * i, j = k0 + e / CP;
      kk[i] = vv[i] = make_uint4(0, 0, 0, 0);
      if (j < n) {
        kk[i] = *reinterpret_cast<const uint4*>(k + j * ld + e % CP * 8);
        vv[i] = *reinterpret_cast<const uint4*>(v + j * ld + e % CP * 8);
      }
    }
    if (k0 > 0) __syncthreads();                     // the previous tile's readers are done
#pragma unroll
    for (int i = 0; i < LN; ++i) {
      const int e = threadIdx.x + 256 * i, at = e / CP * RB + e % CP * 8;
      *reinterpret_cast<uint4*>(kt + at) = kk[i];
      *reinterpret_cast<uint4*>(vt + at) = vv[i];
    }
    __syncthreads();
    if (!live) continue;
    const int tiles = min(4, (n - k0 + 15) / 16);    // sixteens of keys
    f32x4 sc[4];
    float mt = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      sc[t] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (t >= tiles) continue;
      f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        Frag kf;
        kf.u = *reinterpret_cast<const uint4*>(kt + (16 * t + c) * RB + 32 * s + 8 * g);
        a = mfma16(kf.v, qf[s].v, a);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (k0 + 16 * t + 4 * g + r < n) sc[t][r] = a[r] * scale_log2;
        mt = fmaxf(mt, sc[t][r]);
      }
    }
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float mn = fmaxf(m, mt), corr = __builtin_amdgcn_exp2f(m - mn);    // the tile's first key is real: mn is finite
    float ls = 0.f;
    Frag pf[2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = t < tiles ? __builtin_amdgcn_exp2f(sc[t][r] - mn) : 0.f;
        ls += p;
        pf[t >> 1].v[4 * (t & 1) + r] = (bf16)p;
      }
    l = l * corr + ls;
    m = mn;
    const bf16* vr = vt + (4 * g + (c >> 2)) * RB + 4 * (c & 3);
#pragma unroll
    for (int i = 0; i < NT; ++i) o[i] *= corr;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (2 * s >= tiles) continue;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        union {
          s16x4 s[2];
          bf16x8 v;
        } a;
        a.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vr + 32 * s * RB + 16 * i));
        a.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vr + (32 * s + 16) * RB + 16 * i));
        o[i] = mfma16(a.v, pf[s].v, o[i]);
      }
    }
  }
  if (qi >= n) return;                               // all four lanes of a query together: their swaps have partners
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const float inv = 1.0f / l;
  bf16* dst = out + ((long)(r0 + qi) * H + h) * D + 8 * (g >> 1) + 16 * (g & 1);
#pragma unroll
  for (int i = 0; i < NT; i += 2) {
    bf16x4 x, y;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = (bf16)(o[i][r] * inv), y[r] = (bf16)(o[i + 1][r] * inv);
    *reinterpret_cast<uint4*>(dst + 16 * i) = pair16(x, y);
  }
}

enum { SMALL_BIAS = 0, SMALL_GELU = 1, SMALL_SLAB = 2 };

// bf16(s + bias) [-> exact GELU] of four adjacent columns
template <int EPI> __device__ __forceinline__ void small_store(const f32x4& s, const bf16* bias, bf16* y) {
  const bf16x4 bv = *reinterpret_cast<const bf16x4*>(bias);
  bf16x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float v = s[r] + (float)bv[r];
    if (EPI == SMALL_GELU) {
      v = (float)(bf16)v;                            // rounded where GEMM-with-bias -> bf16 -> GELU rounds
      v = gelu_erf(v);
    }
    o[r] = (bf16)v;
  }
  *reinterpret_cast<bf16x4*>(y) = o;
}

// Up to 32 rows: grid (16 W rows, -, slices of K), MF tiles of 16 tokens.  Eight waves fetch both operands of 256 UN of K at a time as the
// matrix instruction reads them and leave them in LDS; then one wave per token tile runs the products as ONE chain over K.  That
// is the order of the LDS ring's sums (gemm_splitk.hip), which takes more rows: a text's embedding is the same bit by bit alone and
// beside others.  Bound by latency: a bge projection has 1 - 5 MB of weights, a few microseconds at HBM rate, and the point is enough
// blocks to ask for them at once.  18 rows, N x K = 2304 x 768: 4.5 us (eight waves that multiply an eighth of K each and add up, in
// another order, 4.1; the 256 x 256 tile kernel 17), 768 x 768 4.2 (3.8), 3072 x 768 4.7 (4.3).
// SLAB: gridDim.z slices of K, slice z's sums to f32 slab z [M, N] (no bias): a long K over few column tiles is 48 blocks that
// each read 100 KB of weights and twice that of X (18 x 768 x 3072: 8.7 us, in four slices 4.8; the norm that adds
// them 3.3 us instead of 2.8).
template <int MF, int EPI, int UN>
__global__ void __launch_bounds__(512) gemm_bias_chain_kernel(const bf16* __restrict__ X, int ldx, const bf16* __restrict__ W, int K,
                                                              void* __restrict__ Yv, int ldy, const bf16* __restrict__ bias, int M, int N) {
  constexpr int CH = 8 * UN;                           // steps of 32 of K at a time
  __shared__ bf16x8 ops[CH][1 + MF][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const int n0 = blockIdx.x * 16, steps = K / 32 / gridDim.z, k0 = blockIdx.z * steps;
  const bf16* wp = W + (long)(n0 + c) * K + 8 * g;
  const bf16* xp[MF];
#pragma unroll
  for (int u = 0; u < MF; ++u) xp[u] = X + (long)min(16 * u + c, M - 1) * ldx + 8 * g;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 v[UN][1 + MF];
  auto fetch = [&](int at) {
#pragma unroll
    for (int i = 0; i < UN; ++i) {
      const int k = min(at + w + 8 * i, steps - 1) + k0;       // no branch: all loads are asked for at once
      v[i][0] = *reinterpret_cast<const bf16x8*>(wp + (long)k * 32);
#pragma unroll
      for (int u = 0; u < MF; ++u) v[i][1 + u] = *reinterpret_cast<const bf16x8*>(xp[u] + (long)k * 32);
    }
  };
  fetch(0);
  for (int at = 0; at < steps; at += CH) {
    if (at > 0) __syncthreads();                       // the products of the steps before are done
#pragma unroll
    for (int i = 0; i < UN; ++i)
#pragma unroll
      for (int u = 0; u <= MF; ++u) ops[w + 8 * i][u][lane] = v[i][u];
    __syncthreads();
    if (at + CH < steps) fetch(at + CH);
    if (w < MF) {
      // operands a group ahead of their products: the chain waits for the matrix pipe only
      const int n = min(CH, steps - at);
      bf16x8 a[2][4], b[2][4];
      auto read = [&](int s, int k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[s][i] = ops[min(k + i, CH - 1)][0][lane], b[s][i] = ops[min(k + i, CH - 1)][1 + w][lane];
      };
      read(0, 0);
#pragma unroll
      for (int k = 0; k < CH; k += 4) {
        if (k + 4 < CH) read((k / 4 + 1) & 1, k + 4);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k + i < n) acc = mfma16(a[(k / 4) & 1][i], b[(k / 4) & 1][i], acc);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  const int m = 16 * w + c, n = n0 + 4 * g;
  if (w >= MF || m >= M) return;
  if constexpr (EPI == SMALL_SLAB) *reinterpret_cast<f32x4*>(static_cast<float*>(Yv) + ((long)blockIdx.z * M + m) * N + n) = acc;
  else small_store<EPI>(acc, bias + n, static_cast<bf16*>(Yv) + (long)m * ldy + n);
}

template <int EPI>
void launch_chain(const void* X, int ldx, const void* W, int K, void* Y, int ldy, const void* bias, int M, int N, int S, hipStream_t st) {
  const dim3 grid(N / 16, 1, S);
  const int un = K / S > 768 ? 4 : (K / S + 255) / 256;
#define CHAIN(MF, UN) \
  if (un == UN && MF == (M <= 16 ? 1 : 2)) \
    gemm_bias_chain_kernel<MF, EPI, UN><<<grid, 512, 0, st>>>((const bf16*)X, ldx, (const bf16*)W, K, Y, ldy, (const bf16*)bias, M, N);
  CHAIN(1, 1) CHAIN(1, 2) CHAIN(1, 3) CHAIN(1, 4) CHAIN(2, 1) CHAIN(2, 2) CHAIN(2, 3) CHAIN(2, 4)
#undef CHAIN
}

// The sizes that neither that kernel nor the ring take: grid (W rows / (16 NF), token tiles of 16 MF), 8 waves that split K in pieces of 32.
// Both operands go from memory straight to registers (W rows and token rows, 64 bytes of a row per four lanes); the
// partial sums meet in LDS.
template <int NF, int MF, int EPI>
__global__ void __launch_bounds__(512) gemm_bias_small_kernel(const bf16* __restrict__ X, int ldx, const bf16* __restrict__ W,
                                                              int K, bf16* __restrict__ Y, int ldy,
                                                              const bf16* __restrict__ bias, int M, int N) {
  constexpr int UN = NF * MF >= 4 ? 3 : 4;
  __shared__ f32x4 red[8][NF * MF][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const int n0 = blockIdx.x * 16 * NF, m0 = blockIdx.y * 16 * MF;
  const bf16* wp[NF];
  const bf16* xp[MF];
#pragma unroll
  for (int f = 0; f < NF; ++f) wp[f] = W + (long)min(n0 + 16 * f + c, N - 1) * K + 8 * g;
#pragma unroll
  for (int u = 0; u < MF; ++u) xp[u] = X + (long)min(m0 + 16 * u + c, M - 1) * ldx + 8 * g;
  f32x4 acc[NF][MF];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int u = 0; u < MF; ++u) acc[f][u] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int kt = K / 32, k1 = kt * (w + 1) / 8;
  int k = kt * w / 8;
  Frag a[UN][NF], b[UN][MF];
  for (; k + UN <= k1; k += UN) {
#pragma unroll
    for (int j = 0; j < UN; ++j) {
#pragma unroll
      for (int f = 0; f < NF; ++f) a[j][f].u = *reinterpret_cast<const uint4*>(wp[f] + (k + j) * 32);
#pragma unroll
      for (int u = 0; u < MF; ++u) b[j][u].u = *reinterpret_cast<const uint4*>(xp[u] + (k + j) * 32);
    }
#pragma unroll
    for (int j = 0; j < UN; ++j)
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int u = 0; u < MF; ++u) acc[f][u] = mfma16(a[j][f].v, b[j][u].v, acc[f][u]);
  }
  for (; k < k1; ++k) {
#pragma unroll
    for (int f = 0; f < NF; ++f) a[0][f].u = *reinterpret_cast<const uint4*>(wp[f] + k * 32);
#pragma unroll
    for (int u = 0; u < MF; ++u) b[0][u].u = *reinterpret_cast<const uint4*>(xp[u] + k * 32);
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int u = 0; u < MF; ++u) acc[f][u] = mfma16(a[0][f].v, b[0][u].v, acc[f][u]);
  }
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int u = 0; u < MF; ++u) red[w][f * MF + u][lane] = acc[f][u];
  __syncthreads();
  for (int it = w; it < NF * MF; it += 8) {
    const int m = m0 + 16 * (it % MF) + c, n = n0 + 16 * (it / MF) + 4 * g;
    if (m >= M || n >= N) continue;
    f32x4 s = red[0][it][lane];
#pragma unroll
    for (int i = 1; i < 8; ++i) s += red[i][it][lane];
    small_store<EPI>(s, bias + n, Y + (long)m * ldy + n);
  }
}

}  // namespace

// qkv [T, ld] bf16: q | k | v of H heads each, D = 64 or 128; cu [texts + 1] row bounds; out [T, H * D]
PENNY_API int penny_encoder_attention(const void* qkv, long ld, const int* cu, int texts, int max_len, int H, int D,
                                      float scale, void* out, hipStream_t stream) {
  if (texts <= 0 || max_len <= 0) return 0;
  if ((D != 64 && D != 128) || H < 1 || H > 65535 || texts > 65535 || ld % 8 || ld < 3L * H * D ||
      ((size_t)qkv | (size_t)out) % 16)
    return (int)hipErrorInvalidValue;
  const dim3 grid((max_len + 63) / 64, H, texts);
  const float s = scale * 1.4426950408889634f;
  if (D == 64) encoder_attention_kernel<64><<<grid, 256, 0, stream>>>((const bf16*)qkv, ld, cu, H, s, (bf16*)out);
  else encoder_attention_kernel<128><<<grid, 256, 0, stream>>>((const bf16*)qkv, ld, cu, H, s, (bf16*)out);
  PENNY_RETURN_LAUNCH();
}

// gemm_splitk.hip
extern "C" int penny_bias_rows_tile(int M, int N, int S);
extern "C" int penny_bias_rows(const void* X, int ldx, const void* W, int K, void* Y, int ldy, const void* bias, int M, int N, int gelu, int slices, int nf,
                               int mt, hipStream_t st);
extern "C" int penny_rows_slabs(const void* X, int ldx, const void* W, int K, float* slabs, int M, int N, int S, int nf, int mt, int paired,
                                hipStream_t st);

namespace {

// Weights whose rows beyond 32 the ring takes
bool ring_shape(int N, int K) { return N >= 16 && N % 16 == 0 && K >= 64 && K % 64 == 0 && (N % 256 == 0 || K <= 1024); }

// Slices of K for the second projection of the feed-forward: as many as bring its blocks near the CUs, 512 of K each at least; 1: not
// split.  By the weight alone, for the same reason: a query embedded beside others would else rank its near-ties otherwise than
// alone, and the prompt that is made of them would miss the prefix cache.  A query of 12 layers of 768 x 3072, us unsplit / in 2 / 3 / 4 / 6: 6
// tokens 422 / 412 / 419 / 414 / 414, 18: 467 / 438 / 437 / 441 / 451, 32: 505 / 472 / 466 / 459 / 466, 48: 599 / 536 / 521 / 511 / 523, 64: 634 / 565 /
// 550 / 545 / 556, 84: 680 / 611 / 623 / 621 / 611, 109: 701 / 627 / 652 / 637 / 640, 179: 743 / 658 / 633 / 669 / 645.  As a call of its own the
// slices' sum is a launch more, so not where K is short: 1024 x 1024 7 rows unsplit 3.7, in 2 slices 5.6, 18: 4.4 / 6.0; 512 x 2048 7: 5.0 / 5.8,
// 18: 6.6 / 6.3; 768 x 3072 7: 6.4 / 6.5, 18: 8.8 / 7.0.
int few_slices(int N, int K) {
  if (K < 3072 || !ring_shape(N, K) || (N != 256 && N != 512 && N != 768 && N != 1024)) return 1;
  int s = 256 / (N / 16);
  if (s > K / 512) s = K / 512;
  while (K % (64 * s)) --s;
  return s;
}

// Parts of K that are summed for themselves and then added in turn, one order of the sums for all numbers of rows: the slices above; of a
// long K that has none the eighths that gemm_bias_small_kernel's waves take (2048 x 8192 7 rows 16.1 us, as one chain 19.5; the ring adds
// them up at no cost); else K is one chain.
int sum_parts(int N, int K) {
  const int s = few_slices(N, K);
  return s > 1 ? s : K > 1024 && K % 512 == 0 && ring_shape(N, K) ? 8 : 1;
}

// The slices as slabs that the next pass adds: up to 192 rows; beyond, the ring adds them itself
int small_slices(int M, int N, int K) { return M <= 192 ? few_slices(N, K) : 1; }

}  // namespace

// The tile (nf | mt << 8) with which a projection goes through the LDS ring of gemm_splitk.hip instead of the kernels above, or 0.
// Blocks of the kernel that splits K read both operands for themselves, which costs more with every further row tile; the ring's tiles share
// them, one round of blocks for all. Us, above (its slices included) or the tile kernel / ring: 2304 x 768 18 rows 4.0 / 4.8, 48 5.5 / 4.8,
// 128 9.3 / 5.8, 256 11.0 / 6.7, 768 20.1 / 11.0, 1536 21.3 / 16.8, 2048 21.6 / 24.8 (two rounds); 768 x 768 48 5.0 / 4.5, 768 10.6 / 6.3, 1536
// 20.2 / 9.0; 3072 x 768 with GELU 128 9.6 / 6.2, 768 24.5 / 15.4, 1024 27.8 / 19.0; 768 x 3072 48 8.6 / 7.0, 192 (in slices,
// on either side, with the launch that adds them) 11.4 / 9.5, 256 (unsplit) 11 / 10.4, 768 35.1 / 15.6, 2048 38.4 / 27.5; 4096 x 1024 512 31.4 / 14.0; 1024 x 4096 128 20.5 / 12.7.  Widths that
// the tile kernel does not take have the library behind them: 1152 x 384 256 4.5 / 4.2, 1024 8.0 / 6.9, 2048 9.5 / 10.2; 384 x 1536 64 - 192 4.9 /
// 6.5: not there.  Nor where K is as long as many rows (2048 x 8192 1000 rows 67.9 / 65.6, 1280 70.0 / 78.3, 2048 79.4 / 90.8).
PENNY_API int penny_bias_rows_plan(int M, int N, int K) {
  if (M <= 32 || !ring_shape(N, K) || M > (N % 256 == 0 ? 2048 : 1024) || (long)M * K > 1 << 23 || small_slices(M, N, K) > 1) return 0;
  return penny_bias_rows_tile(M, N, 1);
}

// Y [M, N] (row stride ldy) = bf16(X W^T + bias) [-> exact GELU]; W [N, K] contiguous; N % 16 == 0, K % 32 == 0, rows in
// whole 16 bytes
PENNY_API int penny_gemm_bias_small(const void* X, int ldx, const void* W, int K, void* Y, int ldy, const void* bias, int M,
                                    int N, int gelu, hipStream_t stream) {
  if (M <= 0) return 0;
  if (N % 16 || K % 32 || ldx % 8 || ldy % 4 || ((size_t)X | (size_t)W) % 16 || ((size_t)Y | (size_t)bias) % 8 ||
      (M + 15) / 16 > 65535)
    return (int)hipErrorInvalidValue;
  const bool sliced = few_slices(N, K) > 1;
  if (M <= 32 && ring_shape(N, K) && (sum_parts(N, K) == 1 || (gelu && sliced))) {
    if (gelu) launch_chain<SMALL_GELU>(X, ldx, W, K, Y, ldy, bias, M, N, 1, stream);
    else launch_chain<SMALL_BIAS>(X, ldx, W, K, Y, ldy, bias, M, N, 1, stream);
    PENNY_RETURN_LAUNCH();
  }
  // (GELU behind a weight of slices: no slabs there, one chain throughout)
  if (const int tile = gelu && M > 32 && small_slices(M, N, K) > 1 ? penny_bias_rows_tile(M, N, 1) : penny_bias_rows_plan(M, N, K))
    return penny_bias_rows(X, ldx, W, K, Y, ldy, bias, M, N, gelu, gelu && sliced ? 1 : sum_parts(N, K), tile & 255, tile >> 8, stream);
#define SMALL(NF, MF)                                                                                                    \
  do {                                                                                                                   \
    const dim3 grid((N + 16 * NF - 1) / (16 * NF), (M + 16 * MF - 1) / (16 * MF));                                       \
    if (gelu)                                                                                                            \
      gemm_bias_small_kernel<NF, MF, SMALL_GELU><<<grid, 512, 0, stream>>>((const bf16*)X, ldx, (const bf16*)W, K,       \
                                                                           (bf16*)Y, ldy, (const bf16*)bias, M, N);      \
    else                                                                                                                 \
      gemm_bias_small_kernel<NF, MF, SMALL_BIAS><<<grid, 512, 0, stream>>>((const bf16*)X, ldx, (const bf16*)W, K,       \
                                                                           (bf16*)Y, ldy, (const bf16*)bias, M, N);      \
  } while (0)
  if (M <= 16) SMALL(1, 1);
  else if (M <= 32) SMALL(1, 2);
  else if (M <= 128) SMALL(1, 4);
  else SMALL(2, 4);
#undef SMALL
  PENNY_RETURN_LAUNCH();
}

namespace {

constexpr int EMBED_ARGS = 960;           // of the 4 KiB that a launch carries

struct EmbedArgs {
  int v[EMBED_ARGS];                      // ids [T] | positions [T] | row bounds [texts + 1]
};

// One wave per token: x = LN(word[id] + bf16(position[p] + type[0])); ids and positions outside their tables give zero rows.
// C4 pieces of 4 values per lane (H = 256 C4), the statistics as in layernorm_wave_kernel.
template <int C4>
__device__ __forceinline__ void embed_row(int row, int id, int p, const bf16* __restrict__ word, int nword,
                                          const bf16* __restrict__ position, int npos, const bf16* __restrict__ type,
                                          const bf16* __restrict__ g, const bf16* __restrict__ b, bf16* __restrict__ y, float eps) {
  constexpr int H = 256 * C4;
  const int lane = threadIdx.x & 63;
  const bool wok = id >= 0 && id < nword, pok = p >= 0 && p < npos;
  const bf16x4* wr = reinterpret_cast<const bf16x4*>(word + (long)(wok ? id : 0) * H);
  const bf16x4* pr = reinterpret_cast<const bf16x4*>(position + (long)(pok ? p : 0) * H);
  const bf16x4* tr = reinterpret_cast<const bf16x4*>(type);
  float v[C4][4], s = 0.f;
#pragma unroll
  for (int c = 0; c < C4; ++c) {
    const bf16x4 wv = wr[lane + 64 * c], pv = pr[lane + 64 * c], tv = tr[lane + 64 * c];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[c][i] = (wok ? (float)wv[i] : 0.f) + (float)(bf16)((pok ? (float)pv[i] : 0.f) + (float)tv[i]);
      s += v[c][i];
    }
  }
  const float mu = wave_sum(s) / (float)H;
  float sq = 0.f;
#pragma unroll
  for (int c = 0; c < C4; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = v[c][i] - mu;
      sq += d * d;
    }
  const float inv = rsqrtf(wave_sum(sq) / (float)H + eps);
#pragma unroll
  for (int c = 0; c < C4; ++c) {
    const bf16x4 gg = reinterpret_cast<const bf16x4*>(g)[lane + 64 * c], bb = reinterpret_cast<const bf16x4*>(b)[lane + 64 * c];
    bf16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (bf16)((v[c][i] - mu) * inv * (float)gg[i] + (float)bb[i]);
    reinterpret_cast<bf16x4*>(y + (long)row * H)[lane + 64 * c] = o;
  }
}

template <int C4>
__global__ void __launch_bounds__(256) encoder_embed_kernel(const int* __restrict__ ids, const int* __restrict__ pos,
                                                            const bf16* __restrict__ word, int nword,
                                                            const bf16* __restrict__ position, int npos,
                                                            const bf16* __restrict__ type, const bf16* __restrict__ g,
                                                            const bf16* __restrict__ b, bf16* __restrict__ y, int T, float eps) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row < T) embed_row<C4>(row, ids[row], pos[row], word, nword, position, npos, type, g, b, y, eps);
}

// The same with ids and positions from the launch's own arguments; the first block leaves the bounds for the launches behind it
template <int C4>
__global__ void __launch_bounds__(256) encoder_embed_args_kernel(EmbedArgs a, const bf16* __restrict__ word, int nword,
                                                                 const bf16* __restrict__ position, int npos,
                                                                 const bf16* __restrict__ type, const bf16* __restrict__ g,
                                                                 const bf16* __restrict__ b, bf16* __restrict__ y, int T, float eps,
                                                                 int* __restrict__ cu, int ncu) {
  const int row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < ncu; i += 256) cu[i] = a.v[2 * T + i];
  if (row < T) embed_row<C4>(row, a.v[row], a.v[T + row], word, nword, position, npos, type, g, b, y, eps);
}

// One wave per text: out[i] = x[cu[i]] / max(|x[cu[i]]|, 1e-12) in f32
__global__ void __launch_bounds__(256) encoder_pool_kernel(const bf16* __restrict__ x, const int* __restrict__ cu, int texts,
                                                           int H, float* __restrict__ out) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= texts) return;
  const bf16* r = x + (long)cu[i] * H;
  float s = 0.f;
  for (int d = lane; d < H; d += 64) s += (float)r[d] * (float)r[d];
  const float n = fmaxf(sqrtf(wave_sum(s)), 1e-12f);
  for (int d = lane; d < H; d += 64) out[(long)i * H + d] = (float)r[d] / n;
}

// One wave per row: y = LN(bf16(sum of the S slabs + bias) + res); H = 256 C4, arithmetic of layernorm_wave_kernel
template <int C4>
__global__ void __launch_bounds__(256) layernorm_slab_kernel(const float* __restrict__ P, int S, const bf16* __restrict__ bias,
                                                             const bf16* __restrict__ res, const bf16* __restrict__ g,
                                                             const bf16* __restrict__ b, bf16* __restrict__ y, int T, float eps) {
  constexpr int H = 256 * C4;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= T) return;
  f32x4 p[C4];
  bf16x4 rv[C4], bv[C4], gg[C4], bb[C4];
#pragma unroll
  for (int c = 0; c < C4; ++c) {
    const int at = lane + 64 * c;
    p[c] = reinterpret_cast<const f32x4*>(P + (long)row * H)[at];
    rv[c] = reinterpret_cast<const bf16x4*>(res + (long)row * H)[at];
    bv[c] = reinterpret_cast<const bf16x4*>(bias)[at];
    gg[c] = reinterpret_cast<const bf16x4*>(g)[at];
    bb[c] = reinterpret_cast<const bf16x4*>(b)[at];
  }
#pragma unroll 4
  for (int i = 1; i < S; ++i)
#pragma unroll
    for (int c = 0; c < C4; ++c) p[c] += reinterpret_cast<const f32x4*>(P + ((long)i * T + row) * H)[lane + 64 * c];
  float v[C4][4], s = 0.f, sq = 0.f;
#pragma unroll
  for (int c = 0; c < C4; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[c][i] = (float)(bf16)(p[c][i] + (float)bv[c][i]) + (float)rv[c][i];
      s += v[c][i];
    }
  const float mu = wave_sum(s) / (float)H;
#pragma unroll
  for (int c = 0; c < C4; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = v[c][i] - mu;
      sq += d * d;
    }
  const float inv = rsqrtf(wave_sum(sq) / (float)H + eps);
#pragma unroll
  for (int c = 0; c < C4; ++c) {
    bf16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (bf16)((v[c][i] - mu) * inv * (float)gg[c][i] + (float)bb[c][i]);
    reinterpret_cast<bf16x4*>(y + (long)row * H)[lane + 64 * c] = o;
  }
}

// y = bf16(sum of the S slabs + bias), four columns per thread
__global__ void __launch_bounds__(256) slab_bias_kernel(const float* __restrict__ P, int S, const bf16* __restrict__ bias,
                                                        bf16* __restrict__ y, int ldy, int M, int N) {
  const int c = N / 4, i = blockIdx.x * 256 + threadIdx.x;
  if (i >= M * c) return;
  const int row = i / c, n = i % c * 4;
  f32x4 p = *reinterpret_cast<const f32x4*>(P + (long)row * N + n);
#pragma unroll 4
  for (int z = 1; z < S; ++z) p += *reinterpret_cast<const f32x4*>(P + ((long)z * M + row) * N + n);
  const bf16x4 bv = *reinterpret_cast<const bf16x4*>(bias + n);
  bf16x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = (bf16)(p[j] + (float)bv[j]);
  *reinterpret_cast<bf16x4*>(y + (long)row * ldy + n) = o;
}

// S = few_slices(N, K) slices of K of X W^T to f32 slabs [S, M, N], up to 192 rows (192 x 1024 and 4 slices: 192 blocks of 4 x 4)
int small_slabs(const void* X, int ldx, const void* W, float* slabs, int S, int M, int N, int K, hipStream_t stream) {
  if (M > 32) {
    const int tile = penny_bias_rows_tile(M, N, S);
    return tile ? penny_rows_slabs(X, ldx, W, K, slabs, M, N, S, tile & 255, tile >> 8, 1, stream) : (int)hipErrorInvalidValue;
  }
  launch_chain<SMALL_SLAB>(X, ldx, W, K, slabs, N, nullptr, M, N, S, stream);
  return (int)hipGetLastError();
}

// y = LN(bf16(X W^T + bias) + res) by slabs
int small_slab_norm(const void* X, const void* W, const void* bias, const void* res, const void* g, const void* b, void* y, float* slabs,
                    int S, int M, int N, int K, float eps, hipStream_t stream) {
  const int rc = small_slabs(X, K, W, slabs, S, M, N, K, stream);
  if (rc) return rc;
#define NORM(C4)                                                                                                        \
  layernorm_slab_kernel<C4><<<(M + 3) / 4, 256, 0, stream>>>(slabs, S, (const bf16*)bias, (const bf16*)res, (const bf16*)g, \
                                                             (const bf16*)b, (bf16*)y, M, eps)
  if (N == 256) NORM(1);
  else if (N == 512) NORM(2);
  else if (N == 768) NORM(3);
  else NORM(4);
#undef NORM
  PENNY_RETURN_LAUNCH();
}

}  // namespace

// ids, pos [T] int32; word [nword, H], position [npos, H], type [>= 1, H], g, b [H], y [T, H] bf16; H = 256, 512, 768 or 1024
PENNY_API int penny_encoder_embed(const int* ids, const int* pos, const void* word, int nword, const void* position, int npos,
                                  const void* type, const void* g, const void* b, void* y, int T, int H, float eps,
                                  hipStream_t stream) {
  if (T <= 0) return 0;
  if (nword < 1 || npos < 1) return (int)hipErrorInvalidValue;
#define EMBED(C4)                                                                                                            \
  encoder_embed_kernel<C4><<<(T + 3) / 4, 256, 0, stream>>>(ids, pos, (const bf16*)word, nword, (const bf16*)position, npos, \
                                                            (const bf16*)type, (const bf16*)g, (const bf16*)b, (bf16*)y, T, eps)
  if (H == 256) EMBED(1);
  else if (H == 512) EMBED(2);
  else if (H == 768) EMBED(3);
  else if (H == 1024) EMBED(4);
  else return (int)hipErrorInvalidValue;
#undef EMBED
  PENNY_RETURN_LAUNCH();
}

// The same for a small batch, meta on the HOST: ids [T] | positions [T] | row bounds [ncu], 2 T + ncu <= 960, which travel with the launch;
// the bounds are left in cu [ncu].  A copy from pageable memory costs 21 us and waits for all work before it, and with it the host's
// lead over the device.  Encodings one after another (waited for singly), us with the copy / here: 6 tokens 398 (440) / 319 (420), 18
// 433 (495) / 334 (452), 128 534 (595) / 420 (572), 10 texts of 40 660 (744) / 554 (727).  The layers as a recorded graph: level (339, 424), 25 us
// less when waited for, and 300 us more the first time of each length.
PENNY_API int penny_encoder_embed_host(const int* meta, int ncu, const void* word, int nword, const void* position, int npos, const void* type,
                                       const void* g, const void* b, void* y, int T, int H, float eps, int* cu, hipStream_t stream) {
  if (T <= 0) return 0;
  if (nword < 1 || npos < 1 || ncu < 0 || T > EMBED_ARGS / 2 || 2 * T + ncu > EMBED_ARGS) return (int)hipErrorInvalidValue;
  EmbedArgs a{};
  for (int i = 0; i < 2 * T + ncu; ++i) a.v[i] = meta[i];
#define EMBED(C4)                                                                                                             \
  encoder_embed_args_kernel<C4><<<(T + 3) / 4, 256, 0, stream>>>(a, (const bf16*)word, nword, (const bf16*)position, npos,    \
                                                                 (const bf16*)type, (const bf16*)g, (const bf16*)b, (bf16*)y, \
                                                                 T, eps, cu, ncu)
  if (H == 256) EMBED(1);
  else if (H == 512) EMBED(2);
  else if (H == 768) EMBED(3);
  else if (H == 1024) EMBED(4);
  else return (int)hipErrorInvalidValue;
#undef EMBED
  PENNY_RETURN_LAUNCH();
}

// x [rows, H] bf16 -> out [texts, H] f32; cu [texts + 1], cu[i] < rows for every text
PENNY_API int penny_encoder_pool(const void* x, const int* cu, int texts, int H, float* out, hipStream_t stream) {
  if (texts <= 0) return 0;
  encoder_pool_kernel<<<(texts + 3) / 4, 256, 0, stream>>>((const bf16*)x, cu, texts, H, out);
  PENNY_RETURN_LAUNCH();
}

PENNY_API int penny_encoder_slices(int T, int H, int F) { return small_slices(T, H, F); }

// penny_gemm_bias_small without GELU by S = penny_encoder_slices(M, N, K) > 1 slices; slabs: f32 [S, M, N].  The sums are those of
// the layers' slab norm.
PENNY_API int penny_gemm_bias_small_split(const void* X, int ldx, const void* W, int K, void* Y, int ldy, const void* bias, int M, int N,
                                          float* slabs, int S, hipStream_t stream) {
  if (M <= 0) return 0;
  if (S < 2 || S != small_slices(M, N, K) || K % 32 || ldx % 8 || ldy % 4 || ((size_t)X | (size_t)W | (size_t)slabs) % 16 ||
      ((size_t)Y | (size_t)bias) % 8)
    return (int)hipErrorInvalidValue;
  const int rc = small_slabs(X, ldx, W, slabs, S, M, N, K, stream);
  if (rc) return rc;
  slab_bias_kernel<<<(M * (N / 4) + 255) / 256, 256, 0, stream>>>(slabs, S, (const bf16*)bias, (bf16*)Y, ldy, M, N);
  PENNY_RETURN_LAUNCH();
}

PENNY_API int penny_layernorm(const void* x, const void* res, const void* g, const void* b, void* y, int T, int H, float eps,
                              int add_residual, hipStream_t stream);

constexpr int PENNY_MISALIGNED = -1;

// All layers of a small batch: x [T, H] bf16 is replaced by the last layer's output.  w: 12 pointers per layer -- qkv, its
// bias, o, its bias, the first norm's weight and bias, fc1, its bias, fc2, its bias, the second norm's weight and bias, each
// contiguous bf16.  ws: T * (6 H + F) bf16, then f32 slabs [penny_encoder_slices(T, H, F), T, H] where that is more than 1.  Shapes as
// penny_gemm_bias_small, penny_encoder_attention and penny_layernorm take them; PENNY_MISALIGNED, and nothing launched, for a weight off
// their 16 bytes (asked here: 144 weights take 18 us in Python).
// The launches of one layer take the host 8 x 2.5 us here and 8 x 7 from Python, where the kernels of a single query
// (18 tokens, 12 layers of 768) run for 440 us in all: 815 -> 497 us for the query.
PENNY_API int penny_encoder_layers(const void* const* w, int layers, void* x, void* ws, const int* cu, int texts, int max_len,
                                   int T, int H, int heads, int F, float eps, float scale, hipStream_t stream) {
  if (T <= 0) return 0;
  if (heads < 1 || H % heads || H % 8 || F % 8) return (int)hipErrorInvalidValue;
  size_t at = 0;
  for (int i = 0; i < 12 * layers; ++i) at |= (size_t)w[i];
  if (at % 16) return PENNY_MISALIGNED;
  bf16* qkv = static_cast<bf16*>(ws);
  bf16 *a = qkv + (long)T * 3 * H, *o = a + (long)T * H, *mid = o + (long)T * H, *h = mid + (long)T * H;
  float* slabs = reinterpret_cast<float*>(h + (long)T * F);
  const int slices = small_slices(T, H, F);
  int rc = 0;
  for (int i = 0; i < layers && rc == 0; ++i, w += 12) {
    rc = penny_gemm_bias_small(x, H, w[0], H, qkv, 3 * H, w[1], T, 3 * H, 0, stream);
    if (rc == 0) rc = penny_encoder_attention(qkv, 3 * H, cu, texts, max_len, heads, H / heads, scale, a, stream);
    if (rc == 0) rc = penny_gemm_bias_small(a, H, w[2], H, o, H, w[3], T, H, 0, stream);
    if (rc == 0) rc = penny_layernorm(o, x, w[4], w[5], mid, T, H, eps, 1, stream);
    if (rc == 0) rc = penny_gemm_bias_small(mid, H, w[6], H, h, F, w[7], T, F, 1, stream);
    if (rc == 0 && slices > 1) {
      rc = small_slab_norm(h, w[8], w[9], mid, w[10], w[11], x, slabs, slices, T, H, F, eps, stream);
    } else {
      if (rc == 0) rc = penny_gemm_bias_small(h, F, w[8], F, o, H, w[9], T, H, 0, stream);
      if (rc == 0) rc = penny_layernorm(o, mid, w[10], w[11], x, T, H, eps, 1, stream);
    }
  }
  return rc;
}
