// BERT / bge encoder (K14) kernels of their own: bidirectional attention straight over the packed QKV rows, and the
// biased projections of small batches.
//
//   penny_encoder_attention   every text attends within itself; texts are short (a query or a transaction: 6 - 128
//                             tokens), so a 64-token tile of one (text, head) is a whole problem and no paged cache is
//                             written first.
//   penny_gemm_bias_small     bf16(x w^T + b) [-> exact GELU] for up to a few hundred rows.
#include "common.h"

namespace {

union Frag {
  uint4 u;
  bf16x8 v;
};

__device__ __forceinline__ f32x4 mfma16(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// grid (query tiles of 64, heads, texts), 4 waves of 16 queries.  qkv [T, ld]: q | k | v, heads side by side.  Per tile of
// 64 keys: S^T = K Q^T with the keys' rows read from memory as operands (the four waves share them in L1), online softmax
// in base 2, O^T += V^T P^T with the value tile transposed in LDS and P straight from the score registers (K slot 8 g + i
// holds keys 4 g + i and 16 + 4 g + i).  Bound by the QKV rows read and the output written: 1024 texts of 6 - 64 tokens
// (36k), 12 heads of 64: 61 us (3.6 TB/s); the paged form took 202 us for the cache write and 72 us for the attention.
template <int D>
__global__ void __launch_bounds__(256) encoder_attention_kernel(const bf16* __restrict__ qkv, long ld,
                                                                const int* __restrict__ cu, int H, float scale_log2,
                                                                bf16* __restrict__ out) {
  constexpr int KS = D / 32, NT = D / 16, LDV = 64 + 8;
  __shared__ __attribute__((aligned(16))) bf16 vt[D * LDV];
  const int r0 = cu[blockIdx.z], n = cu[blockIdx.z + 1] - r0, t0 = blockIdx.x * 64;
  if (t0 >= n) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15, h = blockIdx.y;
  const bf16* q = qkv + (long)r0 * ld + h * D;
  const bf16* k = q + H * D;
  const bf16* v = k + H * D;
  const int qi = t0 + 16 * w + c;
  Frag qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s].u = *reinterpret_cast<const uint4*>(q + min(qi, n - 1) * ld + 32 * s + 8 * g);
  f32x4 o[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const bool live = t0 + 16 * w < n;                 // this wave has a query
  for (int k0 = 0; k0 < n; k0 += 64) {
    Frag kf[4][KS], vv[D / 64][2][1];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s)
        kf[t][s].u = *reinterpret_cast<const uint4*>(k + min(k0 + 16 * t + c, n - 1) * ld + 32 * s + 8 * g);
    // value tile: a thread moves a pair of keys x 8 dims (zeros behind the text's end)
#pragma unroll
    for (int i = 0; i < D / 64; ++i) {
      const int e = threadIdx.x + 256 * i, jp = e / (D / 8), d = e % (D / 8) * 8;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int j = k0 + 2 * jp + r;
        vv[i][r][0].u = *reinterpret_cast<const uint4*>(v + min(j, n - 1) * ld + d);
        if (j >= n) vv[i][r][0].u = make_uint4(0, 0, 0, 0);
      }
    }
    if (k0 > 0) __syncthreads();                     // the previous tile's readers are done
#pragma unroll
    for (int i = 0; i < D / 64; ++i) {
      const int e = threadIdx.x + 256 * i, jp = e / (D / 8), d = e % (D / 8) * 8;
#pragma unroll
      for (int x = 0; x < 8; ++x)
        *reinterpret_cast<bf16x2*>(vt + (d + x) * LDV + 2 * jp) = bf16x2{vv[i][0][0].v[x], vv[i][1][0].v[x]};
    }
    __syncthreads();
    if (!live) continue;
    f32x4 sc[4];
    float mt = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      sc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) sc[t] = mfma16(kf[t][s].v, qf[s].v, sc[t]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[t][r] = k0 + 16 * t + 4 * g + r < n ? sc[t][r] * scale_log2 : -INFINITY;
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
        const float p = __builtin_amdgcn_exp2f(sc[t][r] - mn);
        ls += p;
        pf[t >> 1].v[4 * (t & 1) + r] = (bf16)p;
      }
    l = l * corr + ls;
    m = mn;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      o[i] *= corr;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bf16* vr = vt + (16 * i + c) * LDV + 32 * s + 4 * g;
        const bf16x4 a0 = *reinterpret_cast<const bf16x4*>(vr), a1 = *reinterpret_cast<const bf16x4*>(vr + 16);
        o[i] = mfma16(bf16x8{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]}, pf[s].v, o[i]);
      }
    }
  }
  if (qi >= n) return;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const float inv = 1.0f / l;
  bf16* dst = out + ((long)(r0 + qi) * H + h) * D + 4 * g;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    bf16x4 x;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = (bf16)(o[i][r] * inv);
    *reinterpret_cast<bf16x4*>(dst + 16 * i) = x;
  }
}

// grid (W rows / (16 NF), token tiles of 16 MF), 8 waves that split K in pieces of 32.  Both operands go from memory
// straight to registers (W rows and token rows, 64 bytes of a row per four lanes); the partial sums meet in LDS.
// Bound by latency: a bge projection has 1 - 5 MB of weights, a few microseconds at HBM rate, and the point is enough
// blocks to ask for them at once.  18 rows, N x K = 2304 x 768: 4.3 us, the 256 x 256 tile kernel 17 us (its 9 tiles split
// K over the idle CUs and meet in a second phase); 768 x 3072: 8 and 32 us.
template <int NF, int MF, bool GELU>
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
    const bf16x4 bv = *reinterpret_cast<const bf16x4*>(bias + n);
    bf16x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = s[r] + (float)bv[r];
      if (GELU) {
        v = (float)(bf16)v;                          // rounded where GEMM-with-bias -> bf16 -> GELU rounds
        v = gelu_erf(v);
      }
      y[r] = (bf16)v;
    }
    *reinterpret_cast<bf16x4*>(Y + (long)m * ldy + n) = y;
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

// Y [M, N] (row stride ldy) = bf16(X W^T + bias) [-> exact GELU]; W [N, K] contiguous; N % 16 == 0, K % 32 == 0, rows in
// whole 16 bytes
PENNY_API int penny_gemm_bias_small(const void* X, int ldx, const void* W, int K, void* Y, int ldy, const void* bias, int M,
                                    int N, int gelu, hipStream_t stream) {
  if (M <= 0) return 0;
  if (N % 16 || K % 32 || ldx % 8 || ldy % 4 || ((size_t)X | (size_t)W) % 16 || ((size_t)Y | (size_t)bias) % 8 ||
      (M + 15) / 16 > 65535)
    return (int)hipErrorInvalidValue;
#define SMALL(NF, MF)                                                                                                    \
  do {                                                                                                                   \
    const dim3 grid((N + 16 * NF - 1) / (16 * NF), (M + 16 * MF - 1) / (16 * MF));                                       \
    if (gelu)                                                                                                            \
      gemm_bias_small_kernel<NF, MF, true><<<grid, 512, 0, stream>>>((const bf16*)X, ldx, (const bf16*)W, K, (bf16*)Y,   \
                                                                     ldy, (const bf16*)bias, M, N);                      \
    else                                                                                                                 \
      gemm_bias_small_kernel<NF, MF, false><<<grid, 512, 0, stream>>>((const bf16*)X, ldx, (const bf16*)W, K, (bf16*)Y,  \
                                                                      ldy, (const bf16*)bias, M, N);                     \
  } while (0)
  if (M <= 16) SMALL(1, 1);
  else if (M <= 32) SMALL(1, 2);
  else if (M <= 128) SMALL(1, 4);
  else SMALL(2, 4);
#undef SMALL
  PENNY_RETURN_LAUNCH();
}
