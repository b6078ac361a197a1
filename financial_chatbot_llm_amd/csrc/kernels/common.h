// Shared device helpers for the gfx950 (CDNA4, MI355X) kernel library.
//
// Conventions used by every kernel in this directory:
//  * wave = 64 lanes; block sizes are multiples of 64.
//  * bf16 tensors are moved 16 B (8 elements) per lane per instruction (uint4), math in f32.
//  * every launcher is `extern "C"`, takes raw device pointers + a hipStream_t, never
//    allocates or synchronises (so it can be captured into a hipGraph), and returns the
//    hipError_t of the launch.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define PENNY_API extern "C" __attribute__((visibility("default")))

// Device-side bounds checks, compiled only into the debug library (PENNY_KERNEL_DEBUG=1 python -m
// financial_chatbot_llm_amd._build --debug -> _lib/libpenny_kernels_debug.so, loaded when
// PENNY_KERNEL_DEBUG=1): print the failing condition and trap at the first bad index, instead of
// an out-of-bounds access that faults somewhere later.  The production library has none of them.
#ifdef PENNY_KERNEL_DEBUG
#include <stdio.h>
#define PENNY_DASSERT(cond)                                                                         \
  do {                                                                                              \
    if (!(cond)) {                                                                                  \
      printf("[penny] device assert failed: %s (%s:%d, block %d thread %d)\n", #cond, __FILE__,     \
             __LINE__, (int)blockIdx.x, (int)threadIdx.x);                                          \
      __builtin_trap();                                                                             \
    }                                                                                               \
  } while (0)
#else
#define PENNY_DASSERT(cond) ((void)0)
#endif

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

static constexpr int WAVE = 64;

__device__ __forceinline__ float bf2f(bf16 x) { return (float)x; }
__device__ __forceinline__ bf16 f2bf(float x) { return (bf16)x; }

// 8 x bf16 <-> uint4 (16 B) helpers
union Pack8 {
  uint4 u;
  bf16x8 v;
  bf16 e[8];
};

__device__ __forceinline__ void unpack8(const uint4& u, float* f) {
  Pack8 p;
  p.u = u;
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = (float)p.e[i];
}

__device__ __forceinline__ uint4 pack8(const float* f) {
  Pack8 p;
#pragma unroll
  for (int i = 0; i < 8; ++i) p.e[i] = (bf16)f[i];
  return p.u;
}

// 8 consecutive outputs of a split-K GEMM (gemm_splitk.hip): the sum of its S f32 slabs (slab
// stride `ss` floats), rounded to bf16 exactly where the unsplit GEMM would round its output.
// A decode step's rows are too few to hide one slab's trip behind another's: up to eight slabs (what
// the splits here come to) are all asked for before the first is added, in the same order.  (With the
// norm's weight and residual in the same trip, the rotary table before the slabs and the attention's
// parts in one, the small launches of a 32-layer decode step: 64 rows 7683 -> 7396 us the step, 16
// rows 4673 -> 4519, one row 3160 -> 3118.)
template <int N>
__device__ __forceinline__ void add8_slabs(const float* __restrict__ p, long ss, f32x4* a, f32x4* b) {
  f32x4 u[N], v[N];
#pragma unroll
  for (int s = 0; s < N; ++s) {
    u[s] = *reinterpret_cast<const f32x4*>(p + s * ss);
    v[s] = *reinterpret_cast<const f32x4*>(p + s * ss + 4);
  }
  *a = u[0], *b = v[0];
#pragma unroll
  for (int s = 1; s < N; ++s) *a += u[s], *b += v[s];
}

__device__ __forceinline__ void load8_slabs(const float* __restrict__ p, int S, long ss, float* o) {
  f32x4 a, b;
  switch (S) {
    case 1: add8_slabs<1>(p, ss, &a, &b); break;
    case 2: add8_slabs<2>(p, ss, &a, &b); break;
    case 3: add8_slabs<3>(p, ss, &a, &b); break;
    case 4: add8_slabs<4>(p, ss, &a, &b); break;
    case 6: add8_slabs<6>(p, ss, &a, &b); break;
    default:
      if (S >= 8) {
        add8_slabs<8>(p, ss, &a, &b);
      } else {
        add8_slabs<5>(p, ss, &a, &b);
      }
#pragma unroll 4
      for (int s = S >= 8 ? 8 : 5; s < S; ++s) {
        a += *reinterpret_cast<const f32x4*>(p + s * ss);
        b += *reinterpret_cast<const f32x4*>(p + s * ss + 4);
      }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    o[j] = (float)(bf16)a[j];
    o[4 + j] = (float)(bf16)b[j];
  }
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Block-wide sum for blockDim.x <= 1024; `scratch` needs blockDim.x/64 floats.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += scratch[i];
  __syncthreads();
  return t;
}

// splitmix64 -> two uniforms in (0, 1); counter-based so results are launch-order independent.
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__device__ __forceinline__ float u01_from_bits(uint32_t b) {
  // 24 random mantissa bits, strictly inside (0, 1)
  return ((float)(b >> 8) + 0.5f) * (1.0f / 16777216.0f);
}

// Gumbel noise of vocabulary entry idx for a row seeded `seed` (K12 and the fused LM-head sampler
// draw the SAME noise, so a row samples the same token on either path for equal logits)
__device__ __forceinline__ float gumbel_noise(unsigned long long seed, int idx) {
  const uint64_t r = mix64(seed ^ (0xD1B54A32D192ED03ull * (uint64_t)(idx + 1)));
  return -__logf(-__logf(u01_from_bits((uint32_t)r)));
}

// running (max value, smallest index on ties) of a Gumbel-max / argmax reduction
__device__ __forceinline__ void better(float& bv, int& bi, float v, int i) {
  if (v > bv || (v == bv && i < bi)) {
    bv = v;
    bi = i;
  }
}

#define PENNY_RETURN_LAUNCH() return (int)hipGetLastError()

// Two 4-column groups of bf16 accumulators, lo = columns 16f + 4g .. +3 and hi = 16(f+1) + 4g .. +3
// in lane row g (= lane >> 4) -> the 8 CONSECUTIVE columns 16f + 8*(g>>1) + 16*(g&1) .. +7 of this
// lane, via v_permlane16_swap (odd lane rows of vdst <-> even lane rows of vsrc): one 16-B store
// instead of two 8-B ones (the epilogue store tail is issue-bound).
__device__ __forceinline__ uint4 pair16(bf16x4 lo, bf16x4 hi) {
  union {
    bf16x4 v;
    uint2 u;
  } a, b;
  a.v = lo;
  b.v = hi;
  const auto x = __builtin_amdgcn_permlane16_swap(a.u.x, b.u.x, false, false);
  const auto y = __builtin_amdgcn_permlane16_swap(a.u.y, b.u.y, false, false);
  return make_uint4(x[0], y[0], x[1], y[1]);
}

// GELU as max(x, 0) - |x| erfc(|x| / sqrt 2) / 2, without branches: erfc(z) = t Q(t) exp(-z^2), t = 1 / (1 + 0.3 z), Q of
// degree 8 fitted to a relative error of 2e-8 over z <= 9.5 (beyond, the result is below the smallest f32).  A third of the
// instructions of x/2 (1 + erff), which a GEMM's epilogue does not hide (36,400 x 3072 x 768: 208 us, with erff 260, the
// product and bias alone 163; from gemm_prefill.hip's table of these results 177), and without its cancellation for negative x:
// relative error 1.5e-6 for |x| < 5, there 5e-2.
__device__ __forceinline__ float gelu_erf(float x) {
  const float t = __builtin_amdgcn_rcpf(fmaf(fabsf(x), 0.2121320366859436f, 1.f));
  float q = -0.06471703946590424f;
  q = fmaf(q, t, 0.24254819750785828f);
  q = fmaf(q, t, -0.25561317801475525f);
  q = fmaf(q, t, 0.2731974720954895f);
  q = fmaf(q, t, -0.046815596520900726f);
  q = fmaf(q, t, 0.10721813142299652f);
  q = fmaf(q, t, 0.07424121350049973f);
  q = fmaf(q, t, 0.08534596860408783f);
  q = fmaf(q, t, 0.08459480851888657f);
  const float e = q * t * __builtin_amdgcn_exp2f(x * x * -0.72134752f);
  return fmaf(-fminf(fabsf(x), 64.f), e, fmaxf(x, 0.f));      // (|x| kept finite beside e = 0: gelu(inf) is inf)
}
