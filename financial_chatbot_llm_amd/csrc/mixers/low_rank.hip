// The second factors of low-rank projections in one launch: A = U_a W_a^T in f32 (a decay's pre-activation) and beside it
// G = U_g W_g^T in the storage type (an output gate), U_a [T, ra] and U_g [T, rg] columns of a stacked projection, ranks of 32 or 64.
// Replaces a conversion to f32 and two products (bf16, 15 rows: three launches of 4.6 us, now one of 5.3; 3453 rows of 2048 + 2048: 38, now 22 us).  Bound by the
// results written.
//
// A wave keeps 64 rows of W in registers and walks token tiles of 16.  With bf16 rows each f32 weight is the sum of three bf16 pieces,
// cut and not rounded (exact: 24 bits of significand), whose products with a bf16 value are exact: three 16x16x32 products take
// the place of eight f32 ones, the sums are f32 either way.  Sums that are not finite are worked out again on the f32 instructions: an
// infinity has no such pieces.
#include "mx_common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct LowRank {
  const void* u[2];       // rows of U_a, U_g (storage type), row stride ldu
  const void* w[2];       // W_a f32 [na, ra], W_g of the storage type [ng, rg]
  void* y[2];             // [T, na] f32, [T, ng] of the storage type
  int n[2];
  int blocks_a;           // column blocks of A (256 columns each), then those of G
  long ldu;
  int T, tiles;           // token tiles of 16 per block
};

union Frag {
  unsigned u[4];
  uint4 q;
  bf16x8 v;
};

__device__ __forceinline__ unsigned uppers(float a, float b) {       // the upper halves of two words side by side
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float rest(float a) { return a - __uint_as_float(__float_as_uint(a) & 0xffff0000u); }

// One of the two products for 64 columns from n0 and the block's tokens.  TW: type of W and of the result, KS: 32s of K.
template <typename T, typename TW, int KS>
__device__ __forceinline__ void low_rank_walk(const LowRank& a, int which, int n0) {
  constexpr bool SPLIT = sizeof(T) == 2 && sizeof(TW) == 4;
  constexpr int PL = SPLIT ? 3 : 1, CH = SPLIT || sizeof(T) == 2 ? 1 : 2;       // pieces of a weight; 16-byte chunks of 32 of K
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15, N = a.n[which], K = 32 * KS;
  const TW* w = static_cast<const TW*>(a.w[which]);
  const T* u = static_cast<const T*>(a.u[which]);
  // a lane's 8 of 32 of K: bf16 rows 8 g .., f32 rows 4 g .. and 16 + 4 g .. (the same for both operands)
  Frag wf[4][KS][PL * CH];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const TW* r = w + (long)min(n0 + 16 * f + c, N - 1) * K;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if constexpr (SPLIT) {
        const f32x4 lo = ldf4(r + 32 * s + 8 * g), hi = ldf4(r + 32 * s + 8 * g + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float x = i < 2 ? lo[2 * i & 3] : hi[2 * i & 3], y = i < 2 ? lo[(2 * i + 1) & 3] : hi[(2 * i + 1) & 3];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            wf[f][s][p].u[i] = uppers(x, y);
            x = rest(x);
            y = rest(y);
          }
        }
      } else {
#pragma unroll
        for (int h = 0; h < CH; ++h) wf[f][s][h].q = *reinterpret_cast<const uint4*>(r + 32 * s + (CH == 1 ? 8 * g : 16 * h + 4 * g));
      }
    }
  }
  const int t0 = blockIdx.y * a.tiles, t1 = min(t0 + a.tiles, (a.T + 15) / 16);
  Frag x[KS][CH], nx[KS][CH];
  auto fetch = [&](Frag (&o)[KS][CH], int t) {
    const T* r = u + (long)min(16 * t + c, a.T - 1) * a.ldu;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int h = 0; h < CH; ++h) o[s][h].q = *reinterpret_cast<const uint4*>(r + 32 * s + (CH == 1 ? 8 * g : 16 * h + 4 * g));
  };
  fetch(x, t0);
  for (int t = t0; t < t1; ++t) {
    fetch(nx, min(t + 1, t1 - 1));
    const int m = 16 * t + c;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const int n = n0 + 16 * f;
      if (n >= N) break;
      f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        if constexpr (SPLIT) {
#pragma unroll
          for (int p = 2; p >= 0; --p) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f][k][p].v, x[k][0].v, s, 0, 0, 0);
        } else {
#pragma unroll
          for (int h = 0; h < CH; ++h) s = mma16<T>(wf[f][k][h].q, x[k][h].q, s);
        }
      }
      if constexpr (SPLIT) {
        bool bad = false;
#pragma unroll
        for (int j = 0; j < 4; ++j) bad |= !(fabsf(s[j]) < INFINITY);
        if (__any(bad)) {
          const TW* wr = w + (long)min(n + c, N - 1) * K + g;
          const T* xr = u + (long)min(m, a.T - 1) * a.ldu + g;
          s = f32x4{0.f, 0.f, 0.f, 0.f};
          for (int k = 0; k < K; k += 4) s = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[k], ldf(xr + k), s, 0, 0, 0);
        }
      }
      if (m < a.T) stf4(static_cast<TW*>(a.y[which]) + (long)m * N + n + 4 * g, s);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int h = 0; h < CH; ++h) x[s][h] = nx[s][h];
  }
}

// grid (column blocks of A, then of G; token chunks), 4 waves of 64 columns
template <typename T, int KA, int KG>
__global__ void __launch_bounds__(256) low_rank_kernel(LowRank a) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((int)blockIdx.x < a.blocks_a) {
    const int n0 = blockIdx.x * 256 + 64 * w;
    if (n0 < a.n[0]) low_rank_walk<T, float, KA>(a, 0, n0);
  } else {
    const int n0 = (blockIdx.x - a.blocks_a) * 256 + 64 * w;
    if (n0 < a.n[1]) low_rank_walk<T, T, KG>(a, 1, n0);
  }
}

}  // namespace

// ua [T, ra], ug [T, rg] (row stride ldu, type dt), wa f32 [na, ra], wg [ng, rg] of type dt -> ya f32 [T, na], yg [T, ng] of type dt; ng = 0: A alone.
// ra, rg 32 or 64; na, ng multiples of 16; rows in whole 16 bytes.
MX_API int mx_low_rank(const void* ua, const void* ug, long ldu, const float* wa, int ra, int na, const void* wg, int rg, int ng, float* ya,
                       void* yg, int dt, int T, hipStream_t st) {
  if (T <= 0) return 0;
  const int es = dt == 1 ? 4 : 2;
  if ((ra != 32 && ra != 64) || na <= 0 || na % 16 || ng < 0 || ng % 16 || (ng > 0 && rg != 32 && rg != 64) || ldu * es % 16 || ldu < ra ||
      (ng > 0 && ldu < rg) || ((size_t)ua | (size_t)wa | (size_t)ya) % 16 || (ng > 0 && ((size_t)ug | (size_t)wg | (size_t)yg) % 16) || T > (1 << 24))
    return (int)hipErrorInvalidValue;
  const int ba = (na + 255) / 256, bg = (ng + 255) / 256, tt = (T + 15) / 16;
  // as many token tiles a block as still leave two blocks for every CU
  int tiles = (int)((long)tt * (ba + bg) / 512);
  tiles = tiles < 1 ? 1 : (tiles > 8 ? 8 : tiles);
  const LowRank a{{ua, ug}, {wa, wg}, {ya, yg}, {na, ng}, ba, ldu, T, tiles};
  const dim3 grid(ba + bg, (tt + tiles - 1) / tiles);
  if (grid.y > 65535) return (int)hipErrorInvalidValue;
#define LOW_RANK(KA, KG) MX_DISPATCH(dt, TT, low_rank_kernel<TT, KA, KG><<<grid, 256, 0, st>>>(a))
  if (ra == 32 && (ng == 0 || rg == 32)) LOW_RANK(1, 1);
  else if (ra == 32) LOW_RANK(1, 2);
  else if (ng == 0 || rg == 64) LOW_RANK(2, 2);
  else LOW_RANK(2, 1);
#undef LOW_RANK
  MX_RETURN_LAUNCH();
}
