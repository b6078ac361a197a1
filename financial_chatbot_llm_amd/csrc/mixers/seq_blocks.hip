// Per-row passes of the sequential (post-norm) layered decoders:
//   * embedding gather plus a hashed token-pair row, with the previous token kept per state slot;
//   * layer norm on a sublayer's OUTPUT fused with the residual add and the rounding of the next
//     GEMM input:  x <- x + LN(m) * w,  m = a  or  m = (RMSnorm(a) * wa + RMSnorm(b) * wb) / 2
//     (two mixers side by side);  without a: out = LN(x) * w (the model's last norm);
//   * gated activations act(s * gate) * (s * up) with an optional scale per row (or act alone);
//   * top-k routing on independent sigmoid (or softmax) scores;
//   * per-head RMS norm with a weight shared by the heads, times an activated gate.
#include "mx_common.h"

namespace {

// grid (ceil(max_len / RT), S), RT rows side by side in a block: bound by the way ids -> rows, which rows one after the other walk once
// each (100 rows of 2048 bf16: eight in turn 12.0 us, a block per row 2.5).  The block of a segment's first row is the only one that
// reads the slot's previous token and the one that replaces it with the segment's last id (its read comes first).  VE: adjacent
// columns per access.
template <typename T, int VE, int RT>
__global__ void __launch_bounds__(256) embed_pairs_kernel(const int* __restrict__ ids, const T* __restrict__ table,
                                                          const T* __restrict__ pairs, long mul_prev, long mul_cur, int buckets,
                                                          int* __restrict__ last_token, const int* __restrict__ cu,
                                                          const int* __restrict__ slot, const int* __restrict__ pos,
                                                          float* __restrict__ out, int W, int V) {
  constexpr int LR = 256 / RT;
  const int s = blockIdx.y, i = blockIdx.x * RT + threadIdx.x / LR;
  const int sl = slot[s];
  const int r0 = cu[s], n = cu[s + 1] - r0;
  if ((int)blockIdx.x * RT >= n) return;
  if (i < n) {
    const long r = r0 + i;
    const int raw = ids[r];
    const int id = raw < 0 ? 0 : (raw >= V ? V - 1 : raw);
    long prow = buckets;
    if (pos[r] != 0) {
      const long prev = i > 0 ? ids[r - 1] : (sl >= 0 ? last_token[sl] : 0);
      prow = (prev * mul_prev + (long)raw * mul_cur) % buckets;
      if (prow < 0) prow += buckets;
    }
    const T* e = table + (long)id * W;
    const T* b = pairs + prow * W;
    for (int c = VE * (threadIdx.x % LR); c < W; c += VE * LR) {
      if constexpr (VE == 4) stf4(out + r * W + c, ldf4(e + c) + ldf4(b + c));
      else out[r * W + c] = ldf(e + c) + ldf(b + c);
    }
  }
  if (blockIdx.x == 0 && sl >= 0) {
    __syncthreads();            // every thread of this block has read the carried token
    if (threadIdx.x == 0) last_token[sl] = ids[r0 + n - 1];
  }
}

// one block per row; the row's m lives in LDS (W floats)
template <typename TA, typename TO>
__global__ void post_norm_kernel(float* __restrict__ x, const TA* __restrict__ a, long sa, const float* __restrict__ wa,
                                 const TA* __restrict__ b, long sb, const float* __restrict__ wb,
                                 const float* __restrict__ w, float eps, TO* __restrict__ out, int W) {
  extern __shared__ float m[];
  __shared__ float scratch[16];
  const long t = blockIdx.x;
  float* xr = x + t * W;
  const float inv_w = 1.0f / (float)W;
  if (a == nullptr) {
    for (int i = threadIdx.x; i < W; i += blockDim.x) m[i] = xr[i];
  } else if (b == nullptr) {
    for (int i = threadIdx.x; i < W; i += blockDim.x) m[i] = ldf(a + t * sa + i);
  } else {
    float sa2 = 0.f, sb2 = 0.f;
    for (int i = threadIdx.x; i < W; i += blockDim.x) {
      const float u = ldf(a + t * sa + i), v = ldf(b + t * sb + i);
      sa2 += u * u;
      sb2 += v * v;
    }
    sa2 = mx_block_sum(sa2, scratch);
    sb2 = mx_block_sum(sb2, scratch);
    const float ka = 1.0f / sqrtf(sa2 * inv_w + eps), kb = 1.0f / sqrtf(sb2 * inv_w + eps);
    for (int i = threadIdx.x; i < W; i += blockDim.x)
      m[i] = 0.5f * (ldf(a + t * sa + i) * ka * wa[i] + ldf(b + t * sb + i) * kb * wb[i]);
  }
  // each thread re-reads only the entries it wrote: no barrier needed around m
  float s1 = 0.f;
  for (int i = threadIdx.x; i < W; i += blockDim.x) s1 += m[i];
  const float mean = mx_block_sum(s1, scratch) * inv_w;
  float s2 = 0.f;
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    const float d = m[i] - mean;
    s2 += d * d;
  }
  const float k = 1.0f / sqrtf(mx_block_sum(s2, scratch) * inv_w + eps);
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    const float y = (m[i] - mean) * k * w[i];
    if (a == nullptr) {
      stf(out + t * W + i, y);
    } else {
      const float v = xr[i] + y;
      xr[i] = v;
      if (out != nullptr) stf(out + t * W + i, v);
    }
  }
}

// The same with the row in registers, by fours, R pieces per thread: one read of every input (2400 rows of 2048 f32 with a
// bf16 addend and copy: 19 us, through LDS element by element 34).
// OPEN: the sublayer outputs are pa and pb (a and b say only which of them there are)
template <typename TA, typename TO, int R, bool OPEN>
__global__ void __launch_bounds__(256) post_norm_vec_kernel(float* __restrict__ x, const TA* __restrict__ a, long sa,
                                                            const float* __restrict__ wa, const TA* __restrict__ b, long sb,
                                                            MxPart pa, MxPart pb,
                                                            const float* __restrict__ wb, const float* __restrict__ w,
                                                            float eps, TO* __restrict__ out, int W) {
  __shared__ float scratch[16];
  const long t = blockIdx.x;
  const float inv_w = 1.0f / (float)W;
  const mx_f32x4 zero = mx_f32x4{0.f, 0.f, 0.f, 0.f};
  mx_f32x4 m[R], xv[R], u[R];
  auto sum4 = [](mx_f32x4 v) { return (v[0] + v[1]) + (v[2] + v[3]); };
#pragma unroll
  for (int c = 0; c < R; ++c) {
    const int i = 4 * (threadIdx.x + 256 * c);
    m[c] = xv[c] = u[c] = zero;
    if (i >= W) continue;
    xv[c] = ldf4(x + t * W + i);
    if (OPEN) {
      m[c] = mx_part4<TA>(pa, t, i);
      if (b != nullptr) u[c] = mx_part4<TA>(pb, t, i);
    } else {
      m[c] = a == nullptr ? xv[c] : ldf4(a + t * sa + i);
      if (b != nullptr) u[c] = ldf4(b + t * sb + i);
    }
  }
  if (b != nullptr) {
    float sa2 = 0.f, sb2 = 0.f;
#pragma unroll
    for (int c = 0; c < R; ++c) {
      sa2 += sum4(m[c] * m[c]);
      sb2 += sum4(u[c] * u[c]);
    }
    sa2 = mx_block_sum(sa2, scratch);
    sb2 = mx_block_sum(sb2, scratch);
    const float ka = 1.0f / sqrtf(sa2 * inv_w + eps), kb = 1.0f / sqrtf(sb2 * inv_w + eps);
#pragma unroll
    for (int c = 0; c < R; ++c) {
      const int i = 4 * (threadIdx.x + 256 * c);
      if (i < W) m[c] = 0.5f * (m[c] * ka * ldf4(wa + i) + u[c] * kb * ldf4(wb + i));
    }
  }
  float s1 = 0.f, s2 = 0.f;
#pragma unroll
  for (int c = 0; c < R; ++c) s1 += sum4(m[c]);
  const float mean = mx_block_sum(s1, scratch) * inv_w;
#pragma unroll
  for (int c = 0; c < R; ++c) {
    if (4 * ((int)threadIdx.x + 256 * c) >= W) continue;
    const mx_f32x4 d = m[c] - mean;
    s2 += sum4(d * d);
  }
  const float k = 1.0f / sqrtf(mx_block_sum(s2, scratch) * inv_w + eps);
#pragma unroll
  for (int c = 0; c < R; ++c) {
    const int i = 4 * (threadIdx.x + 256 * c);
    if (i >= W) continue;
    mx_f32x4 y = (m[c] - mean) * k * ldf4(w + i);
    if (a != nullptr) {
      y += xv[c];
      stf4(x + t * W + i, y);
    }
    if (out != nullptr) stf4(out + t * W + i, y);
  }
}

// 0.5 z (1 + tanh(u)) with u = sqrt(2/pi) (z + 0.044715 z^3), written as z sigmoid(2u): one exponential
__device__ __forceinline__ float mx_gelu_tanh(float z) {
  return z * mx_sigmoid(1.5957691216057308f * (z + 0.044715f * z * z * z));
}

__device__ __forceinline__ float mx_act(float v, int act) {
  switch (act) {
    case 1: return mx_silu(v);
    case 2: return mx_gelu_tanh(v);
    case 3: return mx_sigmoid(v);
    default: return v;
  }
}

template <typename T>
__global__ void glu_act_kernel(const T* __restrict__ gate, long sg, const T* __restrict__ up, long su,
                               const float* __restrict__ row_scale, int act, T* __restrict__ out, long so, int n,
                               long total) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long t = i / n;
    const int c = (int)(i - t * n);
    const float s = row_scale != nullptr ? row_scale[t] : 1.0f;
    const float g = mx_act(s * ldf(gate + t * sg + c), act);
    stf(out + t * so + c, up != nullptr ? g * (s * ldf(up + t * su + c)) : g);
  }
}

// the same with 16-byte accesses: grid (rows, column chunks), V elements per thread; every row start and the
// column count are multiples of V elements
template <typename T, int V>
__global__ void glu_act_vec_kernel(const T* __restrict__ gate, long sg, const T* __restrict__ up, long su,
                                   const float* __restrict__ row_scale, int act, T* __restrict__ out, long so, int nv) {
  typedef T vec __attribute__((ext_vector_type(V)));
  const long t = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= nv) return;
  const float s = row_scale != nullptr ? row_scale[t] : 1.0f;
  const vec g = *reinterpret_cast<const vec*>(gate + t * sg + (long)c * V);
  vec u, o;
  if (up != nullptr) u = *reinterpret_cast<const vec*>(up + t * su + (long)c * V);
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const float a = mx_act(s * (float)g[e], act);
    o[e] = (T)(up != nullptr ? a * (s * (float)u[e]) : a);
  }
  *reinterpret_cast<vec*>(out + t * so + (long)c * V) = o;
}

// one wave per token: the `top` largest scores (ties: the lower index) with the score as weight.
// sigmoid scores (1) keep the order of the logits; softmax scores are normalised over all E entries (0)
// or over the chosen entries only (2).
__global__ void route_scores_kernel(const float* __restrict__ z, int E, int top, int sigmoid_scores,
                                    float* __restrict__ outw, int* __restrict__ outi, int T) {
  const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= T) return;
  const float* zr = z + (long)t * E;
  float m = -INFINITY, inv = 1.f;
  if (sigmoid_scores == 0) {
    for (int e = lane; e < E; e += 64) m = fmaxf(m, zr[e]);
    m = mx_wave_max(m);
    float s = 0.f;
    for (int e = lane; e < E; e += 64) s += expf(zr[e] - m);
    inv = 1.0f / mx_wave_sum(s);
  }
  unsigned long long taken_lo = 0, taken_hi = 0;     // this lane's entries already chosen (E <= 64 * 128)
  for (int k = 0; k < top; ++k) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int e = lane, j = 0; e < E; e += 64, ++j) {
      const bool used = j < 64 ? (taken_lo >> j) & 1 : (taken_hi >> (j - 64)) & 1;
      if (used) continue;
      const float c = zr[e];
      if (c > bv || (c == bv && e < bi) || bi == 0x7fffffff) {
        bv = c;
        bi = e;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (oi != 0x7fffffff && (bi == 0x7fffffff || ov > bv || (ov == bv && oi < bi))) {
        bv = ov;
        bi = oi;
      }
    }
    if (bi != 0x7fffffff && (bi & 63) == lane) {
      const int j = bi >> 6;
      if (j < 64) taken_lo |= 1ull << j; else taken_hi |= 1ull << (j - 64);
    }
    if (lane == 0) {
      const int e = bi == 0x7fffffff ? 0 : bi;
      outi[(long)t * top + k] = e;
      outw[(long)t * top + k] = bi == 0x7fffffff ? 0.f : (sigmoid_scores == 1 ? mx_sigmoid(zr[e])
                                : sigmoid_scores == 2 ? zr[e] : expf(zr[e] - m) * inv);
    }
  }
  if (sigmoid_scores == 2 && lane == 0) {       // softmax over the chosen logits (the first is the largest)
    float* w = outw + (long)t * top;
    const float m2 = w[0];
    float s = 0.f;
    for (int k = 0; k < top; ++k) {
      w[k] = expf(w[k] - m2);
      s += w[k];
    }
    const float r = 1.0f / s;
    for (int k = 0; k < top; ++k) w[k] *= r;
  }
}

// grid (rows, H): head h's P outputs / rms * w[P] * act(gate); w null: no weight
template <typename TI, typename TG, typename TO>
__global__ void head_norm_gate_kernel(const TI* __restrict__ in, long si, const float* __restrict__ w, float eps,
                                      const TG* __restrict__ gate, long sg, int act, TO* __restrict__ out, int P) {
  __shared__ float scratch[16];
  const long t = blockIdx.x;
  const int h = blockIdx.y, H = gridDim.y;
  const TI* r = in + t * si + (long)h * P;
  float ss = 0.f;
  for (int i = threadIdx.x; i < P; i += blockDim.x) {
    const float v = ldf(r + i);
    ss += v * v;
  }
  ss = mx_block_sum(ss, scratch);
  const float k = 1.0f / sqrtf(ss / (float)P + eps);
  for (int i = threadIdx.x; i < P; i += blockDim.x)
    stf(out + (t * H + h) * P + i,
        ldf(r + i) * k * (w != nullptr ? w[i] : 1.f) * mx_act(ldf(gate + t * sg + (long)h * P + i), act));
}

// The same by fours with L lanes per head (4 L >= P): 2400 rows of 16 heads of 128 15 us, one block per head 30
template <typename TI, typename TG, typename TO, int L>
__global__ void __launch_bounds__(256) head_norm_gate_vec_kernel(const TI* __restrict__ in, long si, const float* __restrict__ w,
                                                                 float eps, const TG* __restrict__ gate, long sg, int act,
                                                                 TO* __restrict__ out, int H, int P, long total) {
  const long id = (long)blockIdx.x * (256 / L) + threadIdx.x / L;
  if (id >= total) return;
  const long t = id / H;
  const int h = (int)(id - t * H), i = 4 * (threadIdx.x % L);
  const bool live = i < P;
  mx_f32x4 v = mx_f32x4{0.f, 0.f, 0.f, 0.f}, z = v;
  if (live) {
    v = ldf4(in + t * si + (long)h * P + i);
    z = ldf4(gate + t * sg + (long)h * P + i);
  }
  float ss = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
#pragma unroll
  for (int o = 1; o < L; o <<= 1) ss += __shfl_xor(ss, o, 64);
  const float k = 1.0f / sqrtf(ss / (float)P + eps);
  if (!live) return;
  v *= k;
  if (w != nullptr) v *= ldf4(w + i);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] *= mx_act(z[e], act);
  stf4(out + id * P + i, v);
}

}  // namespace

MX_API int mx_embed_pairs(const int* ids, const void* table, const void* pairs, int dt, int mul_prev, int mul_cur,
                          int buckets, int* last_token, const int* cu, const int* slot, const int* pos, float* out,
                          int S, int max_len, int W, int V, hipStream_t st) {
  if (S <= 0 || max_len <= 0) return 0;
  if (buckets < 1) return (int)hipErrorInvalidValue;
  // a row to a block up to 16384 blocks, beyond eight (500 rows beside 511 single ones: 57 and 12 us)
  const bool wide = W % 4 == 0 && ((size_t)table | (size_t)pairs) % (dt == 1 ? 16 : 8) == 0 && (size_t)out % 16 == 0;
  const bool one = (long)max_len * S <= 16384;
#define EMBED(VE, RT)                                                                                                     \
  MX_DISPATCH(dt, TT, embed_pairs_kernel<TT, VE, RT><<<dim3((max_len + RT - 1) / RT, S), 256, 0, st>>>(                    \
      ids, (const TT*)table, (const TT*)pairs, mul_prev, mul_cur, buckets, last_token, cu, slot, pos, out, W, V))
  if (wide && one) EMBED(4, 1);
  else if (wide) EMBED(4, 8);
  else if (one) EMBED(1, 1);
  else EMBED(1, 8);
#undef EMBED
  MX_RETURN_LAUNCH();
}

// x f32 [T, W].  a given: x <- x + LN(m) * w in place and, with out, out = x in type dt_out;
// m = a, or with b: (RMSnorm(a) wa + RMSnorm(b) wb) / 2 (a, b of type dt_ab, row strides sa, sb).
// a null: out = LN(x) * w.
MX_API int mx_post_norm(float* x, const void* a, long sa, const float* wa, const void* b, long sb, const float* wb,
                        int dt_ab, const float* w, float eps, void* out, int dt_out, int T, int W, hipStream_t st) {
  if (T <= 0) return 0;
  if ((size_t)W * sizeof(float) > 60 * 1024 || (a == nullptr && out == nullptr)) return (int)hipErrorInvalidValue;
  // in registers up to 4096 values: 32 a thread leave too few blocks in flight (4096 rows of 8192: 120 us, through LDS 88)
  if (W % 4 == 0 && W > 0 && W <= 4096 && ((size_t)x | (size_t)w | (size_t)wa | (size_t)wb) % 16 == 0 &&
      (a == nullptr || mx_by_four(a, sa, dt_ab)) && (b == nullptr || (a != nullptr && mx_by_four(b, sb, dt_ab))) &&
      mx_by_four(out, W, dt_out)) {
#define POST_NORM(R)                                                                                                     \
  MX_DISPATCH(dt_ab, TA, MX_DISPATCH(dt_out, TO, post_norm_vec_kernel<TA, TO, R, false><<<T, 256, 0, st>>>(              \
      x, (const TA*)a, sa, wa, (const TA*)b, sb, MxPart{}, MxPart{}, wb, w, eps, (TO*)out, W)))
    if (W <= 1024) POST_NORM(1);
    else if (W <= 2048) POST_NORM(2);
    else POST_NORM(4);
#undef POST_NORM
    MX_RETURN_LAUNCH();
  }
  const int nt = W >= 1024 ? 512 : 256;
  MX_DISPATCH(dt_ab, TA, MX_DISPATCH(dt_out, TO, post_norm_kernel<TA, TO><<<T, nt, (size_t)W * sizeof(float), st>>>(
      x, (const TA*)a, sa, wa, (const TA*)b, sb, wb, w, eps, (TO*)out, W)));
  MX_RETURN_LAUNCH();
}

// The same for sublayer outputs that are still apart (b may be null).  W and all rows in whole fours, W <= 4096.
MX_API int mx_post_norm_parts(float* x, const MxPart* a, const float* wa, const MxPart* b, const float* wb, int dt_ab, const float* w,
                              float eps, void* out, int dt_out, int T, int W, hipStream_t st) {
  if (T <= 0) return 0;
  if (a == nullptr || W <= 0 || W % 4 || W > 4096 || !mx_part_by_four(*a, dt_ab) ||
      (b != nullptr && (!mx_part_by_four(*b, dt_ab) || wa == nullptr || wb == nullptr)) || w == nullptr ||
      ((size_t)x | (size_t)w | (size_t)wa | (size_t)wb) % 16 || !mx_by_four(out, W, dt_out))
    return (int)hipErrorInvalidValue;
  const MxPart pb = b != nullptr ? *b : MxPart{};
#define POST_NORM(R)                                                                                                     \
  MX_DISPATCH(dt_ab, TA, MX_DISPATCH(dt_out, TO, post_norm_vec_kernel<TA, TO, R, true><<<T, 256, 0, st>>>(               \
      x, (const TA*)a, 0, wa, (const TA*)b, 0, *a, pb, wb, w, eps, (TO*)out, W)))
  if (W <= 1024) POST_NORM(1);
  else if (W <= 2048) POST_NORM(2);
  else POST_NORM(4);
#undef POST_NORM
  MX_RETURN_LAUNCH();
}

// act: 1 SiLU, 2 tanh-form GeLU; up null: the activation alone
MX_API int mx_glu_act(const void* gate, long sg, const void* up, long su, const float* row_scale, int act, void* out,
                      long so, int dt, int T, int n, hipStream_t st) {
  const long total = (long)T * n;
  if (total <= 0) return 0;
  const int V = dt == 1 ? 4 : 8;                       // elements per 16 bytes
  const bool aligned = n % V == 0 && sg % V == 0 && so % V == 0 && (up == nullptr || su % V == 0) &&
                       ((size_t)gate | (size_t)out | (size_t)up) % 16 == 0 && (size_t)n / V <= 65535u * 256u;
  if (aligned) {
    const int nv = n / V;
    dim3 grid(T, (nv + 255) / 256);
    if (dt == 1)
      glu_act_vec_kernel<float, 4><<<grid, 256, 0, st>>>((const float*)gate, sg, (const float*)up, su, row_scale, act,
                                                         (float*)out, so, nv);
    else
      glu_act_vec_kernel<bf16, 8><<<grid, 256, 0, st>>>((const bf16*)gate, sg, (const bf16*)up, su, row_scale, act,
                                                        (bf16*)out, so, nv);
    MX_RETURN_LAUNCH();
  }
  const int blocks = (int)((total + 255) / 256 < 16384 ? (total + 255) / 256 : 16384);
  MX_DISPATCH(dt, TT, glu_act_kernel<TT><<<blocks, 256, 0, st>>>((const TT*)gate, sg, (const TT*)up, su, row_scale, act,
                                                                  (TT*)out, so, n, total));
  MX_RETURN_LAUNCH();
}

MX_API int mx_route_scores(const float* z, int E, int top, int sigmoid_scores, float* outw, int* outi, int T,
                           hipStream_t st) {
  if (T <= 0) return 0;
  if (E > 64 * 128 || top > E) return (int)hipErrorInvalidValue;
  route_scores_kernel<<<(T + 3) / 4, 256, 0, st>>>(z, E, top, sigmoid_scores, outw, outi, T);
  MX_RETURN_LAUNCH();
}

// in [T, H*P] (row stride si, type dt_in), gate [T, H*P] slice (row stride sg, type dt_gate), out [T, H*P]
// contiguous of type dt_out; w f32 [P] or null; act: 1 SiLU, 3 sigmoid
MX_API int mx_head_norm_gate(const void* in, long si, int dt_in, const float* w, float eps, const void* gate, long sg,
                             int dt_gate, int act, void* out, int dt_out, int T, int H, int P, hipStream_t st) {
  if (T <= 0) return 0;
  // by four with several heads to a block from 2^18 values on; a block per head is the sooner done for less (16 heads of 128, us:
  // 64 rows 3.2, by four 3.4, 256 rows 4.4 and 3.6)
  if (P % 4 == 0 && P > 0 && P <= 256 && (long)T * H * P >= 1 << 18 && mx_by_four(in, si, dt_in) && mx_by_four(gate, sg, dt_gate) &&
      mx_by_four(out, P, dt_out) && (size_t)w % 16 == 0 && (long)T * H < (1L << 31)) {
    const long total = (long)T * H;
#define HEAD_NORM(L)                                                                                                      \
  MX_DISPATCH(dt_in, TI, MX_DISPATCH(dt_gate, TG, MX_DISPATCH(dt_out, TO, head_norm_gate_vec_kernel<TI, TG, TO, L>        \
      <<<(unsigned)((total + 256 / L - 1) / (256 / L)), 256, 0, st>>>((const TI*)in, si, w, eps, (const TG*)gate, sg, act, \
                                                                      (TO*)out, H, P, total))))
    if (P <= 64) HEAD_NORM(16);
    else if (P <= 128) HEAD_NORM(32);
    else HEAD_NORM(64);
#undef HEAD_NORM
    MX_RETURN_LAUNCH();
  }
  const int nt = P >= 256 ? 256 : (P > 64 ? 128 : 64);
  dim3 grid(T, H);
  MX_DISPATCH(dt_in, TI, MX_DISPATCH(dt_gate, TG, MX_DISPATCH(dt_out, TO, head_norm_gate_kernel<TI, TG, TO>
      <<<grid, nt, 0, st>>>((const TI*)in, si, w, eps, (const TG*)gate, sg, act, (TO*)out, P))));
  MX_RETURN_LAUNCH();
}
