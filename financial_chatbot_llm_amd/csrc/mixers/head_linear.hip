// A matrix per head on rows of heads, in place: y[t, h, :] = W[h] x[t, h, :], x a strided view (a part of each head's query, say),
// y contiguous [T, H, N] -- the key up-projection folded into the queries of latent attention, and its value up-projection.  A
// batched library product wants the heads outside, which cost a copy of its own on both sides.
//
// A block owns 16 MF tokens of one head; its four waves take the output columns by 32 (two operand rows groups of 16 as A: a lane's
// four sums are adjacent columns of one token), and both operands go from memory straight to registers: a head's matrix is 48 KB,
// read from L2 and shared by a block's waves in L1.  Bound by the rows of y, x and by latency in small steps.
#include "mx_common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// The sums of row groups f0 and f1 (neighbours, or the same at the end) for token t of head h, as this lane holds them
template <typename T>
__device__ __forceinline__ void put_pair(T* dst, int g, bool both, const f32x4& s0, const f32x4& s1) {
  typedef T vec4 __attribute__((ext_vector_type(4)));
  vec4 lo, hi;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    lo[r] = (T)s0[r];
    hi[r] = (T)s1[r];
  }
  if constexpr (sizeof(T) == 2) {
    if (both) {                              // eight adjacent columns per lane
      union {
        vec4 v;
        uint2 u;
      } a, b;
      a.v = lo;
      b.v = hi;
      const auto q0 = __builtin_amdgcn_permlane16_swap(a.u.x, b.u.x, false, false);
      const auto q1 = __builtin_amdgcn_permlane16_swap(a.u.y, b.u.y, false, false);
      *reinterpret_cast<uint4*>(dst + 8 * (g >> 1) + 16 * (g & 1)) = make_uint4(q0[0], q1[0], q0[1], q1[1]);
      return;
    }
  }
  *reinterpret_cast<vec4*>(dst + 4 * g) = lo;
  if (both) *reinterpret_cast<vec4*>(dst + 16 + 4 * g) = hi;
}

template <typename T, int MF>
__global__ void __launch_bounds__(256) head_linear_kernel(const T* __restrict__ x, long sxt, long sxh, const T* __restrict__ w,
                                                          T* __restrict__ y, int Tn, int H, int N, int K) {
  constexpr int ES = sizeof(T);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, col = lane & 15;
  const int h = blockIdx.y, t0 = blockIdx.x * 16 * MF, nt = N / 16, ks = K * ES / 64;
  const char* xp[MF];
#pragma unroll
  for (int u = 0; u < MF; ++u)
    xp[u] = reinterpret_cast<const char*>(x + (long)min(t0 + 16 * u + col, Tn - 1) * sxt + h * sxh) + 16 * g;
  const char* wh = reinterpret_cast<const char*>(w + (long)h * N * K) + 16 * g;
  for (int p = wv; 2 * p < nt; p += 4) {
    const int f0 = 2 * p, f1 = min(f0 + 1, nt - 1);
    const char* w0 = wh + (long)(16 * f0 + col) * K * ES;
    const char* w1 = wh + (long)(16 * f1 + col) * K * ES;
    f32x4 acc[2][MF];
#pragma unroll
    for (int u = 0; u < MF; ++u) acc[0][u] = acc[1][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = 0; k < ks; ++k) {
      const uint4 a0 = *reinterpret_cast<const uint4*>(w0 + 64 * k), a1 = *reinterpret_cast<const uint4*>(w1 + 64 * k);
      uint4 b[MF];
#pragma unroll
      for (int u = 0; u < MF; ++u) b[u] = *reinterpret_cast<const uint4*>(xp[u] + 64 * k);
#pragma unroll
      for (int u = 0; u < MF; ++u) {
        acc[0][u] = mma16<T>(a0, b[u], acc[0][u]);
        acc[1][u] = mma16<T>(a1, b[u], acc[1][u]);
      }
    }
#pragma unroll
    for (int u = 0; u < MF; ++u) {
      const int t = t0 + 16 * u + col;
      if (t >= Tn) continue;                 // with all lanes of its row groups: the swaps stay among live ones
      put_pair<T>(y + ((long)t * H + h) * N + 16 * f0, g, f1 > f0, acc[0][u], acc[1][u]);
    }
  }
}

// Many tokens: a block's 64 go to LDS, whole rows at a time, and the waves take pairs of row groups for all of them.  Read
// straight from memory as above a load of 16 rows touches 16 lines for its 1 KB, and the tokens' loads, which every wave and pair
// repeated, were the L1's work.  LDS rows are 16 bytes longer than K, so that 16 of them start in different banks.
template <typename T>
__global__ void __launch_bounds__(256) head_linear_tile_kernel(const T* __restrict__ x, long sxt, long sxh, const T* __restrict__ w,
                                                               T* __restrict__ y, int Tn, int H, int N, int K) {
  extern __shared__ __attribute__((aligned(16))) char xs[];
  constexpr int ES = sizeof(T), MF = 4;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, col = lane & 15;
  const int h = blockIdx.y, t0 = blockIdx.x * 16 * MF, nt = N / 16, ks = K * ES / 64, cpr = K * ES / 16, rb = K * ES + 16;
  for (int e = threadIdx.x; e < 16 * MF * cpr; e += 256) {
    const int r = e / cpr, ch = e - r * cpr;
    *reinterpret_cast<uint4*>(xs + r * rb + 16 * ch) =
        *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(x + (long)min(t0 + r, Tn - 1) * sxt + h * sxh) + 16 * ch);
  }
  __syncthreads();
  const char* xp = xs + col * rb + 16 * g;
  const char* wh = reinterpret_cast<const char*>(w + (long)h * N * K) + 16 * g;
  for (int p = wv; 2 * p < nt; p += 4) {
    const int f0 = 2 * p, f1 = min(f0 + 1, nt - 1);
    const char* w0 = wh + (long)(16 * f0 + col) * K * ES;
    const char* w1 = wh + (long)(16 * f1 + col) * K * ES;
    f32x4 acc[2][MF];
#pragma unroll
    for (int u = 0; u < MF; ++u) acc[0][u] = acc[1][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = 0; k < ks; ++k) {
      const uint4 a0 = *reinterpret_cast<const uint4*>(w0 + 64 * k), a1 = *reinterpret_cast<const uint4*>(w1 + 64 * k);
#pragma unroll
      for (int u = 0; u < MF; ++u) {
        const uint4 b = *reinterpret_cast<const uint4*>(xp + 16 * u * rb + 64 * k);
        acc[0][u] = mma16<T>(a0, b, acc[0][u]);
        acc[1][u] = mma16<T>(a1, b, acc[1][u]);
      }
    }
#pragma unroll
    for (int u = 0; u < MF; ++u) {
      const int t = t0 + 16 * u + col;
      if (t >= Tn) continue;
      put_pair<T>(y + ((long)t * H + h) * N + 16 * f0, g, f1 > f0, acc[0][u], acc[1][u]);
    }
  }
}

}  // namespace

// x [T, H, K] (strides sxt, sxh elements, whole 16 bytes), w [H, N, K] contiguous, y [T, H, N] contiguous, all of type dt;
// N % 16 == 0, rows of w and x in whole 64 bytes.  Blocks of 64 tokens share a head's matrix better, blocks of 16 are four times as
// many.  Us, bf16, 16 heads, batched product and copies / by 16 / by 64 tokens: 256 x 96: 64 tokens 9.6 / 3.7 / 6.1, 200: 15.7 / 3.8 /
// 6.2, 600: 15.2 / 6.7 / 6.7, 2500: 32.9 / 18.4 / 15.8, 5065: 50.1 / 33.5 / 25.0; 96 x 256: 64: 10.5 / 3.9 / 6.3, 600: 16.8 / 8.2 / 6.6, 5065:
// 45.8 / 45.9 / 24.7; f32 256 x 96: 64: 12.4 / 6.3 / 11.8, 600: 28.9 / 15.9 / 13.9, 5065: 81 / 88 / 64; 8 heads: 600 11.3 / 5.0 / 6.3, 1200
// 15.1 / 7.0 / 6.7.  By 64 with the tokens in LDS, against straight from memory: 256 x 96 600 6.6 / 5.4, 1200 10.5 / 7.2, 5065 24.7 / 17.0;
// 96 x 256 600 6.6 / 5.9, 2500 16.5 / 10.6, 5065 25.3 / 21.4; 8 heads 5065 16.7 / 10.0; f32 256 x 96 600 13.3 / 13.5, 5065 68 / 57.  Rows
// of more than a kilobyte stay out of LDS (f32 96 x 256 by 32 tokens there: 600 13.5 / 14.6, 5065 66 / 66).
MX_API int mx_head_linear(const void* x, long sxt, long sxh, const void* w, void* y, int T, int H, int N, int K, int dt,
                          hipStream_t st) {
  if (T <= 0 || H <= 0) return 0;
  const int es = dt == 1 ? 4 : 2;
  if (N < 16 || N % 16 || K < 1 || K * es % 64 || sxt * es % 16 || sxh * es % 16 || ((size_t)x | (size_t)w | (size_t)y) % 16 || H > 65535)
    return (int)hipErrorInvalidValue;
  const int rb = K * es + 16;
  if ((long)T * H > 8192 && 64 * rb <= 65536)
    MX_DISPATCH(dt, TT, head_linear_tile_kernel<TT><<<dim3((T + 63) / 64, H), 256, 64 * rb, st>>>((const TT*)x, sxt, sxh, (const TT*)w,
                                                                                                   (TT*)y, T, H, N, K));
  else if ((long)T * H > 8192)
    MX_DISPATCH(dt, TT, head_linear_kernel<TT, 4><<<dim3((T + 63) / 64, H), 256, 0, st>>>((const TT*)x, sxt, sxh, (const TT*)w, (TT*)y, T,
                                                                                         H, N, K));
  else
    MX_DISPATCH(dt, TT, head_linear_kernel<TT, 1><<<dim3((T + 15) / 16, H), 256, 0, st>>>((const TT*)x, sxt, sxh, (const TT*)w, (TT*)y, T,
                                                                                         H, N, K));
  MX_RETURN_LAUNCH();
}
