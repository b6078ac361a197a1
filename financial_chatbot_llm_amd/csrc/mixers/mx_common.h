// Shared helpers of the sequence-mixer kernel library (gfx950): state-space and matrix-state scans,
// latent and windowed attention, top-k routing and the 32-bit residual stream of the layered decoders.
//
// Conventions: wave = 64 lanes; every launcher is `extern "C"`, takes raw device pointers and a
// hipStream_t, never allocates or synchronises (hipGraph-capturable) and returns the launch's
// hipError_t.  Activations come in two storage types chosen by a run-time code (0: bf16,
// 1: f32); all arithmetic is f32.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define MX_API extern "C" __attribute__((visibility("default")))
#define MX_RETURN_LAUNCH() return (int)hipGetLastError()

typedef __bf16 bf16;

template <typename T> __device__ __forceinline__ float ldf(const T* p);
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ldf<bf16>(const bf16* p) { return (float)*p; }
template <typename T> __device__ __forceinline__ void stf(T* p, float v);
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void stf<bf16>(bf16* p, float v) { *p = (bf16)v; }

// run BODY with T bound to the storage type of code `dt`
#define MX_DISPATCH(dt, T, ...)        \
  do {                                 \
    if ((dt) == 1) {                   \
      using T = float;                 \
      __VA_ARGS__;                     \
    } else {                           \
      using T = bf16;                  \
      __VA_ARGS__;                     \
    }                                  \
  } while (0)

__device__ __forceinline__ float mx_wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ float mx_wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// block-wide sum, blockDim.x <= 1024; scratch: 16 floats of LDS
__device__ __forceinline__ float mx_block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = mx_wave_sum(v);
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += scratch[i];
  __syncthreads();
  return t;
}

__device__ __forceinline__ float mx_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float mx_silu(float x) { return x * mx_sigmoid(x); }
// softplus without a clamp: log(1 + e^x), evaluated so that neither tail overflows
__device__ __forceinline__ float mx_softplus(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

// factor on the accumulated values of a softmax with running maximum m and sum l: 1 / l, or with a sink
// exp(m) / (exp(m) l + exp(sink)) evaluated from the larger exponent down
__device__ __forceinline__ float mx_softmax_scale(float m, float l, const float* sink, int h) {
  if (sink == nullptr) return 1.0f / l;
  const float sk = sink[h], M = fmaxf(m, sk);
  const float f = expf(m - M);
  return f / (l * f + expf(sk - M));
}

// D += A B of a 16 x 16 tile over 64 bytes of K per row: a 16-byte operand is 8 bf16 (one 16x16x32 product) or 4 f32 (four
// 16x16x4 products, step j taking K element 4 g + j of both sides)
typedef float mx_f32x4 __attribute__((ext_vector_type(4)));
template <typename T> __device__ __forceinline__ mx_f32x4 mma16(uint4 a, uint4 b, mx_f32x4 c);
template <> __device__ __forceinline__ mx_f32x4 mma16<bf16>(uint4 a, uint4 b, mx_f32x4 c) {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  union { uint4 u; v8 v; } x, y;
  x.u = a;
  y.u = b;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.v, y.v, c, 0, 0, 0);
}
template <> __device__ __forceinline__ mx_f32x4 mma16<float>(uint4 a, uint4 b, mx_f32x4 c) {
  union { uint4 u; mx_f32x4 v; } x, y;
  x.u = a;
  y.u = b;
#pragma unroll
  for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x.v[j], y.v[j], c, 0, 0, 0);
  return c;
}

// four neighbouring elements, as f32
__device__ __forceinline__ mx_f32x4 ldf4(const float* p) { return *reinterpret_cast<const mx_f32x4*>(p); }
__device__ __forceinline__ mx_f32x4 ldf4(const bf16* p) {
  typedef bf16 v4 __attribute__((ext_vector_type(4)));
  const v4 x = *reinterpret_cast<const v4*>(p);
  return mx_f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
}
template <typename T> __device__ __forceinline__ void stf4(T* p, mx_f32x4 x) {
  typedef T v4 __attribute__((ext_vector_type(4)));
  *reinterpret_cast<v4*>(p) = v4{(T)x[0], (T)x[1], (T)x[2], (T)x[3]};
}
// what a launch reads or writes once and nobody needs before much else has passed (recurrent states): not kept in the caches
__device__ __forceinline__ mx_f32x4 ldf4_once(const float* p) { return __builtin_nontemporal_load(reinterpret_cast<const mx_f32x4*>(p)); }
__device__ __forceinline__ void stf4_once(float* p, mx_f32x4 x) { __builtin_nontemporal_store(x, reinterpret_cast<mx_f32x4*>(p)); }
// rows of `stride` elements of type code dt (1: f32) may be read and written by four
inline bool mx_by_four(const void* p, long stride, int dt) { return stride % 4 == 0 && (size_t)p % (dt == 1 ? 16 : 8) == 0; }

// A sublayer's output as the norm behind it reads it, so that what would only add it up needs no launch of its own (a step of 64 rows:
// the sum of a product's K slices 4.4 us, of a token's experts 4.9): rows p [T, ld] of the storage type, `slabs` f32 slices of K of them
// (slab elements apart, their sum rounded to the type), or nothing (p null); with top > 0 a token's routed rows besides, added to those in
// turn: row pos[t, k] of ys times wts[t, k] (null: 1), or for an entry idx[t, k] >= E the token's own row of h.  The order of
// the sums and the roundings are those of the launches that write it out.
struct MxPart {
  const void* p;
  long ld, slab;
  const void* ys;
  long sy;
  const int* pos;
  const int* idx;
  const float* wts;
  const void* h;
  long sh;
  int slabs, E, top;
};
// columns c .. c + 3 of row t
template <typename T> __device__ __forceinline__ mx_f32x4 mx_part4(const MxPart& a, long t, int c) {
  mx_f32x4 v = mx_f32x4{0.f, 0.f, 0.f, 0.f};
  if (a.slabs > 0) {
    const float* p = static_cast<const float*>(a.p) + t * a.ld + c;
    v = ldf4(p);
    for (int s = 1; s < a.slabs; s += 4) {                 // four loads at a time
      mx_f32x4 u[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) u[j] = ldf4(p + min(s + j, a.slabs - 1) * a.slab);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (s + j < a.slabs) v += u[j];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (float)(T)v[e];
  } else if (a.p != nullptr) {
    v = ldf4(static_cast<const T*>(a.p) + t * a.ld + c);
  }
  if (a.top == 0) return v;
  for (int k = 0; k < a.top; k += 4) {
    mx_f32x4 u[4];
    float w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const long i = t * a.top + min(k + j, a.top - 1);
      w[j] = k + j < a.top ? (a.wts != nullptr ? a.wts[i] : 1.f) : 0.f;
      u[j] = ldf4(a.idx[i] >= a.E ? static_cast<const T*>(a.h) + t * a.sh + c : static_cast<const T*>(a.ys) + a.pos[i] * a.sy + c);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (w[j] != 0.f)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += w[j] * u[j][e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = (float)(T)v[e];
  return v;
}
// rows of it may be read by four (type code dt)
inline bool mx_part_by_four(const MxPart& a, int dt) {
  return mx_by_four(a.p, a.ld, a.slabs > 0 ? 1 : dt) && a.slab % 4 == 0 && a.slabs >= 0 && (a.slabs == 0 || a.p != nullptr) &&
         (a.top == 0 || (a.top > 0 && a.pos != nullptr && a.idx != nullptr && mx_by_four(a.ys, a.sy, dt) && mx_by_four(a.h, a.sh, dt)));
}

// A token whose value is not finite must not reach the tokens before it through the zeros of a triangular factor: such
// elements of a tile (rows 4 g + r of column lane % 16) become zero, and the first one's row is returned (16: none).
__device__ __forceinline__ int mx_drop_nonfinite(mx_f32x4& x, int g) {
  bool bad = false;
#pragma unroll
  for (int r = 0; r < 4; ++r) bad |= !(fabsf(x[r]) < INFINITY);
  if (!__any(bad)) return 16;
  int first = 16;
#pragma unroll
  for (int r = 3; r >= 0; --r)
    if (!(fabsf(x[r]) < INFINITY)) {
      first = 4 * g + r;
      x[r] = 0.f;
    }
  first = min(first, __shfl_xor(first, 16, 64));
  return min(first, __shfl_xor(first, 32, 64));
}

// Blocks numbered over the tiles of `tile` rows that the segments have: block id's segment and its first row there, or false.
// per > 0: every segment has that many blocks, the longest segment's tiles.  In a step of prompts and single rows most of those
// would be empty and the live ones meet on few CUs (prompts of 540, 300 and 327 rows beside 21 single rows: an attention's 34 x
// 4 x 24 blocks, 376 of them live, did 31 us of work per CU in 65 us), so with per = 0 the tiles are numbered one segment after the
// other (rows / tile + S of them at most) and found by a scan of the row counts, 64 lanes with NL segments each at a time.
template <int NL>
__device__ __forceinline__ bool mx_tile_scan(const int* __restrict__ cu, int S, int tile, int id, int& s, int& t0) {
  const int lane = threadIdx.x & 63;
  for (int base = 0; base < S; base += 64 * NL) {
    int c[NL + 1], tiles[NL], sum = 0;
#pragma unroll
    for (int k = 0; k <= NL; ++k) c[k] = cu[min(base + NL * lane + k, S)];
#pragma unroll
    for (int k = 0; k < NL; ++k) sum += tiles[k] = (c[k + 1] - c[k] + tile - 1) / tile;
    int upto = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(upto, o, 64);
      if (lane >= o) upto += x;
    }
    const unsigned long long past = __ballot(upto > id);
    if (past == 0) {
      id -= __builtin_amdgcn_readlane(upto, 63);
      continue;
    }
    const int at = __ffsll(past) - 1, first = base + NL * at;
    id -= __builtin_amdgcn_readlane(upto - sum, at);
    s = first;
#pragma unroll
    for (int k = 0; k < NL - 1; ++k) {                       // of the lane's segments the one that holds the block
      const int t = __builtin_amdgcn_readlane(tiles[k], at);
      if (s == first + k && id >= t) id -= t, ++s;
    }
    t0 = id * tile;
    return true;
  }
  return false;
}
// NL: 4 shortens the scan's chain (a window's 1,024 segments 130.7 -> 121.4 us, 4,096 of them 717 -> 538), 1 has the fewer instructions
// (convolutions, whose blocks are many and short: 512 segments 30.7 us, with 4 32.5).
template <int NL>
__device__ __forceinline__ bool mx_tile_place(const int* __restrict__ cu, int S, int per, int tile, int id, int& s, int& t0) {
  if (per > 0) {
    s = per == 1 ? id : id / per;
    if (s >= S) return false;
    t0 = (id - s * per) * tile;
    return t0 < cu[s + 1] - cu[s];
  }
  return S <= 64 ? mx_tile_scan<1>(cu, S, tile, id, s, t0) : mx_tile_scan<NL>(cu, S, tile, id, s, t0);
}

// Blocks per segment, or 0 for the scan: where the longest segment's tiles for every segment are no more blocks than the scan's
// (segments alike, or as short as a tile), a block finds its place without it.  (32 segments of 5 rows, tiles of 16: an attention
// in f32 28.6 -> 20.3 us.)  Beside very many segments empty blocks are cheaper than the scan, up to slack S / 1024 of the scan's blocks
// in all, by the kernel's work per block: 1,023 single rows and a prompt of 64, convolution 52.5 us by the scan, 37.7 so; 2,047 and 130
// 125 and 69, their window attention 270 and 206; 511 and 64 25.7 and 23.6; convolved heads of 1,023 and 20 42 and 30, 100 43 and 50.
inline int mx_tile_per(int S, int rows, int max_len, int tile, int slack = 0) {
  long per = ((long)max_len + tile - 1) / tile;
  const long scan = (long)S + rows / tile;
  if (per * S <= scan) return (int)per;
  per |= 1;                              // single rows' only tiles, every 2nd or 4th or 8th block, would meet on a few XCDs
  return per * S <= scan + scan * S * slack / 1024 ? (int)per : 0;
}
inline int mx_tile_count(int S, int rows, int max_len, int tile, int slack = 0) {
  const int per = mx_tile_per(S, rows, max_len, tile, slack);
  return per > 0 ? per * S : S + rows / tile;
}

constexpr int PAGE_ROWS = 64;            // tokens per cache page

// The parts that several blocks left of one (row, head)'s attention, ws [rows, H, nsplit, P + 2]: unnormalised values, running maximum and
// sum (sigm: plain sums of independently weighted values).  grid (rows, H), a thread per value.  Bound by latency: every
// load is asked for at once, the maxima and sums of 64 parts by a lane each (as three loops over the parts, 17 rows of 8 heads of 256 took 8.9 us
// and 22 of 16 of 128 6.3; now 4.6 and 4.8, 78 of 16 7.4 and 4.0).
template <typename T>
__global__ void attend_merge_kernel(const float* __restrict__ ws, const T* __restrict__ gate, long sgate, int gate_elem,
                                    const float* __restrict__ sink, T* __restrict__ out, int H, int P, int nsplit, int sigm) {
  const long row = blockIdx.x;
  const int h = blockIdx.y, lane = threadIdx.x & 63, r = threadIdx.x;
  const float* w = ws + (row * H + h) * nsplit * (long)(P + 2);
  float m, l;
  auto stats = [&](int from) {             // of the 64 parts from there on
    const float* part = w + (long)min(from + lane, nsplit - 1) * (P + 2) + P;
    m = from + lane < nsplit && !sigm ? part[0] : -INFINITY;
    l = part[1];
  };
  stats(0);
  const float sk = sink != nullptr ? sink[h] : -INFINITY;
  const float gh = gate != nullptr && !gate_elem ? ldf(gate + row * sgate + h) : 0.f;
  const float ge = gate != nullptr && gate_elem && r < P ? ldf(gate + row * sgate + (long)h * P + r) : 0.f;
  constexpr int B = 8;
  float v[B];
  auto load = [&](int b) {
#pragma unroll
    for (int i = 0; i < B; ++i) v[i] = w[(long)min(b + i, nsplit - 1) * (P + 2) + min(r, P - 1)];
  };
  load(0);
  float M = fmaxf(mx_wave_max(m), sk);
  if (nsplit > 64) {
    for (int from = 64; from < nsplit; from += 64) {
      stats(from);
      M = fmaxf(M, mx_wave_max(m));
    }
    stats(0);
  }
  float e = m != -INFINITY ? expf(m - M) : 0.f;
  auto of = [](float x, int i) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), i)); };
  float L = sink != nullptr ? expf(sk - M) : 0.f, a = 0.f;      // the sink counts once, not once per part
  for (int b = 0; b < nsplit; b += B) {
    if (b > 0) load(b);
    if (b > 0 && b % 64 == 0) {
      stats(b);
      e = m != -INFINITY ? expf(m - M) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < B; ++i) {
      if (b + i >= nsplit) break;
      const int at = (b + i) & 63;
      if (sigm) {
        a += v[i];
      } else if (of(m, at) != -INFINITY) {
        L += of(l, at) * of(e, at);
        a += v[i] * of(e, at);
      }
    }
  }
  float f = sigm ? 1.0f : 1.0f / L;
  if (gate != nullptr && !gate_elem) f *= mx_sigmoid(gh);
  if (r < P) stf(out + (row * H + h) * P + r, a * f * (gate != nullptr && gate_elem ? mx_sigmoid(ge) : 1.0f));
}
template <typename T>
inline void attend_merge(const float* ws, const T* gate, long sgate, int gate_elem, const float* sink, T* out, int rows, int H, int P,
                         int nsplit, int sigm, hipStream_t st) {
  attend_merge_kernel<T><<<dim3(rows, H), (P + 63) / 64 * 64, 0, st>>>(ws, gate, sgate, gate_elem, sink, out, H, P, nsplit, sigm);
}

// tanh with one division and no branch.  |z| < 0.6: the fifth convergent of Lambert's continued fraction
// z / (1 + z^2 / (3 + z^2 / (5 + ...))), relative error below 1e-8 there; beyond: (1 - e) / (1 + e), e = exp(-2|z|)
__device__ __forceinline__ float mx_tanh(float z) {
  const float a = fabsf(z), q = z * z;
  const bool small = a < 0.6f;
  const float e = __expf(-2.0f * a);
  const float num = small ? a * (945.0f + q * (105.0f + q)) : 1.0f - e;
  const float den = small ? 945.0f + q * (420.0f + 15.0f * q) : 1.0f + e;
  return copysignf(num / den, z);
}
