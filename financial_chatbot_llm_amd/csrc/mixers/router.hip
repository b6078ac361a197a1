// The router of a routed feed-forward in one launch: logits z = W h (+ b) in f32, scores and the `top` choice, for up to 64
// experts (identity ones among them).  Before: a conversion of h to f32, a library product and the choice, three launches.
//
// Two forms, chosen by the rows of the step:
//   rows   one or four tokens per block; a quarter of the block's threads shares a quarter of the experts and splits K, the sums
//          of a wave meet by lane exchanges that halve the experts a lane holds.  Bound by latency (one round of loads, the
//          exchanges, the choice) and by the router's bytes, which every block reads from L2.
//   tile   16 tokens per block on the f32 matrix cores, 8 waves split K, the partial sums meet in LDS.  Bound by the f32 products.
// Either way products and sums are f32 and the choice runs on one lane per expert, by rank (ties: the lower index).
// The clamped unit of a shared expert's gate and up columns, which needs nothing of the router, may run in blocks behind the router's: a launch
// less for work that fits beside a kernel that waits for latency (gezavik, four such layers: 17 rows 552 -> 541 us, 64 1275 -> 1265, 130 mixed 1040 -> 1015).
#include "mx_common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Most tokens of the rows form, by one and by four per block.  Every block reads all of W, so the kernel's time grows with E x W and
// the library's hardly does; the rule of the calls that come here is ops.mixers.router_takes.  Us, conversion, library product and
// choice / here, W in the memory-side cache, 34 experts of width 2048, bf16: 1 token 15.7 / 10.2, 64: 17.4 / 10.6, 256: 18.3 / 10.9, 512: 19.7 /
// 14.6, 1024: 22.5 / 14.9, 2048: 27.8 / 18.8, 5000: 36.6 / 30.2, 16000: 82.6 / 49.9 (in a decode step, W from HBM, 64 tokens take 13.9); f32 64: 13.5 / 10.3,
// 1024: 15.4 / 12.5.  8 of 2048: 64: 17.6 / 4.5, 5000: 33.5 / 14.3; 32 of 8192: 64: 34.5 / 16.1, 5000: 84 / 79; 48 of 4096: 64: 19.6 / 16.2, 1024:
// 29.5 / 23.3, 5000: 51 / 60; f32 64: 17.0 / 15.6, 1024: 17.6 / 19.3; 48 of 8192 64: 25 / 27.  64 of 2048: 64: 17.4 / 15.5, 512 (by four, whose sums no
// longer fit the registers): 19.5 / 33.4, 2048: 30.9 / 27.6, 5000: 41 / 46; f32 64: 14.8 / 15.9; of 1024: 64: 16.9 / 11.6, 5000: 32.8 / 30.8; f32 64: 12.3 /
// 12.0; of 4096: 64: 19.8 / 22.2.
constexpr int ROWS_1 = 256, ROWS_4 = 1024;

enum { ROUTE_SOFTMAX = 0, ROUTE_SIGMOID = 1, ROUTE_SOFTMAX_TOP = 2 };

struct Router {
  const void* h;          // [T, W], row stride ldh
  long ldh;
  const float* w;         // [E, W]
  const float* zbias;     // on the logits, or null
  const float* bias;      // on the scores for the choice alone (biased), or null
  int biased;             // choose by score + bias (0: by the logits)
  int score, renorm;
  float wscale;
  int E, top, W, T;
  float* outw;
  int* outi;
  // blocks from `blocks` on: out = unit(gate, up), rows of nv 16-byte pieces
  int blocks;
  const void *gate, *up;
  long sgate, sup;
  float limit, alpha;
  void* out;
  int nv;
};

// glu_clamp_vec_kernel's values, a piece of 16 bytes per thread
template <typename T> __device__ __forceinline__ void router_glu(const Router& a) {
  constexpr int V = 16 / sizeof(T);
  typedef T vec __attribute__((ext_vector_type(V)));
  const long i = (long)(blockIdx.x - a.blocks) * blockDim.x + threadIdx.x, t = i / a.nv;
  const int c = (int)(i - t * a.nv);
  if (t >= a.T) return;
  const vec gv = *reinterpret_cast<const vec*>(static_cast<const T*>(a.gate) + t * a.sgate + (long)c * V);
  const vec uv = *reinterpret_cast<const vec*>(static_cast<const T*>(a.up) + t * a.sup + (long)c * V);
  vec o;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const float g = fminf((float)gv[e], a.limit);
    const float u = fminf(fmaxf((float)uv[e], -a.limit), a.limit);
    o[e] = (T)(g * mx_sigmoid(a.alpha * g) * (u + 1.0f));
  }
  *reinterpret_cast<vec*>(static_cast<T*>(a.out) + (t * a.nv + c) * V) = o;
}

// The choice of one token by one wave: z is lane e's logit (e < E).  An entry's rank is the number of those before it: larger,
// or equal with a lower index; what is not a number comes last.
__device__ __forceinline__ void route_choose(const Router& a, float z, long t) {
  const int lane = threadIdx.x & 63, E = a.E;
  const bool in = lane < E;
  float s = z;                                           // ROUTE_SOFTMAX_TOP: of the chosen logits, below
  if (a.score == ROUTE_SIGMOID) {
    s = mx_sigmoid(z);
  } else if (a.score == ROUTE_SOFTMAX) {
    const float m = mx_wave_max(in ? z : -INFINITY), x = in ? expf(z - m) : 0.f;
    s = x * (1.0f / mx_wave_sum(x));
  }
  const float c = a.biased ? s + (a.bias != nullptr && in ? a.bias[lane] : 0.f) : z;
  const bool nan = c != c;
  int rank = 0;
  for (int j = 0; j < E; ++j) {
    const float cj = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(c), j));
    rank += (cj > c || (cj == c && j < lane) || (nan && (cj == cj || j < lane))) ? 1 : 0;
  }
  const bool mine = in && rank < a.top;
  if (a.score == ROUTE_SOFTMAX_TOP) {
    const float m = mx_wave_max(mine ? z : -INFINITY), x = mine ? expf(z - m) : 0.f;
    s = x * (1.0f / mx_wave_sum(x));
  }
  if (a.biased && nan) s = 0.f;
  float f = a.wscale;
  if (a.renorm) f = a.wscale / (mx_wave_sum(mine ? s : 0.f) + 1e-20f);
  if (mine) {
    a.outw[t * a.top + rank] = s * f;
    a.outi[t * a.top + rank] = a.biased && nan ? 0 : lane;
  }
}

// lanes l and l ^ 32 (16): x of one with y of the other, summed: the lower half ends with x's sum, the upper with y's
__device__ __forceinline__ float halve32(float x, float y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float halve16(float x, float y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int O> __device__ __forceinline__ float halve(float x, float y) {
  const bool up = threadIdx.x & O;
  return (up ? y : x) + __shfl_xor(up ? x : y, O, 64);
}

// 1024 threads, TB tokens.  Four groups of 256 threads take EP experts each (4 EP: the experts rounded up to 16), a thread every
// 256th four K elements of all tokens.
template <typename T, int EP, int TB>
__global__ void __launch_bounds__(1024) router_rows_kernel(Router a) {
  __shared__ float part[TB][4][4][16];                       // token, group, wave, expert of the group
  if ((int)blockIdx.x >= a.blocks) return router_glu<T>(a);
  const long t0 = (long)blockIdx.x * TB;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = threadIdx.x >> 8;
  const T* h[TB];
#pragma unroll
  for (int i = 0; i < TB; ++i) h[i] = static_cast<const T*>(a.h) + min(t0 + i, (long)a.T - 1) * a.ldh;
  float acc[TB][16];
#pragma unroll
  for (int i = 0; i < TB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  for (int k = (threadIdx.x & 255) * 4; k < a.W; k += 1024) {
    f32x4 x[TB], r[EP];
#pragma unroll
    for (int e = 0; e < EP; ++e) r[e] = ldf4(a.w + (long)min(q * EP + e, a.E - 1) * a.W + k);
#pragma unroll
    for (int i = 0; i < TB; ++i) x[i] = ldf4(h[i] + k);
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
      for (int e = 0; e < EP; ++e)
        acc[i][e] = fmaf(x[i][3], r[e][3], fmaf(x[i][2], r[e][2], fmaf(x[i][1], r[e][1], fmaf(x[i][0], r[e][0], acc[i][e]))));
  }
#pragma unroll
  for (int i = 0; i < TB; ++i) {                             // lanes 4 e .. 4 e + 3 end with expert e's sum
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < EP) acc[i][e] = halve32(acc[i][e], acc[i][e + 8]);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[i][e] = halve16(acc[i][e], acc[i][e + 4]);
#pragma unroll
    for (int e = 0; e < 2; ++e) acc[i][e] = halve<8>(acc[i][e], acc[i][e + 2]);
    float z = halve<4>(acc[i][0], acc[i][1]);
    z += __shfl_xor(z, 2, 64);
    z += __shfl_xor(z, 1, 64);
    if ((lane & 3) == 0) part[i][q][w & 3][lane >> 2] = z;
  }
  __syncthreads();
  if (w >= TB || t0 + w >= a.T) return;
  float z = 0.f;
  if (lane < a.E) {
    const int gq = lane / EP, e = lane % EP;
    z = (part[w][gq][0][e] + part[w][gq][1][e]) + (part[w][gq][2][e] + part[w][gq][3][e]);
    if (a.zbias != nullptr) z += a.zbias[lane];
  }
  route_choose(a, z, t0 + w);
}

// 512 threads, 16 tokens; NF groups of 16 experts
template <typename T, int NF>
__global__ void __launch_bounds__(512, 4) router_tile_kernel(Router a) {
  __shared__ f32x4 red[8][NF][64];
  __shared__ float zt[16][16 * NF + 1];
  if ((int)blockIdx.x >= a.blocks) return router_glu<T>(a);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15, t0 = blockIdx.x * 16;
  const T* h = static_cast<const T*>(a.h) + (long)min(t0 + c, a.T - 1) * a.ldh + 8 * g;
  const float* r[NF];
  f32x4 acc[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    r[f] = a.w + (long)min(16 * f + c, a.E - 1) * a.W + 8 * g;
    acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int kt = a.W / 32, k1 = kt * (w + 1) / 8;
#pragma unroll 2
  for (int k = kt * w / 8; k < k1; ++k) {
    const f32x4 x0 = ldf4(h + 32 * k), x1 = ldf4(h + 32 * k + 4);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const f32x4 w0 = ldf4(r[f] + 32 * k), w1 = ldf4(r[f] + 32 * k + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(w0[j], x0[j], acc[f], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[j], x1[j], acc[f], 0, 0, 0);
    }
  }
#pragma unroll
  for (int f = 0; f < NF; ++f) red[w][f][lane] = acc[f];
  __syncthreads();
  if (w < NF) {
    f32x4 s = red[0][w][lane];
#pragma unroll
    for (int v = 1; v < 8; ++v) s += red[v][w][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) zt[c][16 * w + 4 * g + i] = s[i];
  }
  __syncthreads();
  for (int i = w; i < 16 && t0 + i < a.T; i += 8) {
    float z = lane < a.E ? zt[i][lane] : 0.f;
    if (a.zbias != nullptr && lane < a.E) z += a.zbias[lane];
    route_choose(a, z, t0 + i);
  }
}

template <typename T, int NF> void router_launch(Router a, hipStream_t st) {
  const int tokens = a.T <= ROWS_1 ? 1 : a.T <= ROWS_4 ? 4 : 16, threads = a.T <= ROWS_4 ? 1024 : 512;
  a.blocks = (a.T + tokens - 1) / tokens;
  const unsigned grid = a.blocks + (unsigned)(((long)a.T * a.nv + threads - 1) / threads);
  if (a.T <= ROWS_1) router_rows_kernel<T, 4 * NF, 1><<<grid, 1024, 0, st>>>(a);
  else if (a.T <= ROWS_4) {
    if constexpr (NF <= 3) router_rows_kernel<T, 4 * NF, 4><<<grid, 1024, 0, st>>>(a);
  } else if constexpr (sizeof(T) == 2) router_tile_kernel<T, NF><<<grid, 512, 0, st>>>(a);
}

}  // namespace

// h [T, W] of type dt (row stride ldh), w f32 [E, W], zbias f32 [E] or null: logits z = w h + zbias.  score: 0 softmax over all
// entries, 1 sigmoid, 2 softmax over the chosen logits.  biased != 0: the largest score + bias (f32 [E] or null) are chosen,
// weighted by the score itself; else the largest logits.  renorm != 0: weights divided by their sum (+ 1e-20); times wscale.
// outw, outi [T, top].  E <= 64, W % 32 == 0, 16-byte rows.  The tile form is for bf16: f32 takes at most ROWS_4 rows.  More than 48
// entries take no rows between ROWS_1 and ROWS_4.  n > 0: act [T, n] = mx_glu_clamp of the columns gate and up besides, all of type dt in whole 16 bytes.
MX_API int mx_router(const void* h, long ldh, int dt, const float* w, const float* zbias, const float* bias, int biased,
                     int score, int renorm, float wscale, int E, int top, int W, float* outw, int* outi, const void* gate, long sgate,
                     const void* up, long sup, float limit, float alpha, void* act, int n, int T, hipStream_t st) {
  if (T <= 0) return 0;
  const int V = dt == 1 ? 4 : 8;
  if (E < 1 || E > 64 || top < 1 || top > E || W < 32 || W % 32 || ldh * (dt == 1 ? 4 : 2) % 16 ||
      ((size_t)h | (size_t)w) % 16 || score < 0 || score > 2 || (biased && score == ROUTE_SOFTMAX_TOP) || (dt == 1 && T > ROWS_4) ||
      (E > 48 && T > ROWS_1 && T <= ROWS_4) || n < 0 || (n > 0 && (n % V || sgate % V || sup % V || ((size_t)gate | (size_t)up | (size_t)act) % 16)) ||
      (long)T * (n / V) > 1L << 36)
    return (int)hipErrorInvalidValue;
  const Router a{h, ldh, w, zbias, bias, biased, score, renorm, wscale, E, top, W, T, outw, outi, 0, gate, up, sgate, sup, limit, alpha, act, n / V};
  MX_DISPATCH(dt, TT, switch ((E + 15) / 16) {
    case 1: router_launch<TT, 1>(a, st); break;
    case 2: router_launch<TT, 2>(a, st); break;
    case 3: router_launch<TT, 3>(a, st); break;
    default: router_launch<TT, 4>(a, st);
  });
  MX_RETURN_LAUNCH();
}
