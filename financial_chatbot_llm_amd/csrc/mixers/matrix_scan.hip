// Token-by-token f32 recurrences over a flat batch of segments (segment s: rows cu[s]..cu[s+1]-1,
// state slot slot[s] (< 0: padding, skipped), zero state when its first row is at position 0).
//
// mx_matrix_scan: a [D, P] state per head with one decay per head and key channel d (acting on row d):
//     gla:    g = sigmoid(a + a_bias)^(1/tau);              S <- g S + k v^T;            o = S^T q
//     delta:  g = exp(-exp(A_log[h]) softplus(a + a_bias));  S <- g S;  u = b (v - S^T k);
//             S <- S + k u^T;  o = S^T q;    q, k unit vectors per head first, b = sigmoid(beta)
//   and q scaled by D^-1/2 in both; or (mx_decay_scan) one FIXED decay per head,
//     fixed:  S <- decay[h] S + act(k) act(v)^T;  o = S^T act(q) * out_scale
//   with the activation (none | SiLU) applied while the rows are staged and no prep launch.  Two launches:
//     prep   one block per token, fully parallel: the decays g (written over `a`), and for the delta
//            rule the unit-norm factors of q and k and sigmoid(beta) (steps of single rows -- decode --
//            skip this launch: the scan's one-token form computes them while it stages the row);
//     scan   column p of S never meets another column, so a lane owns RPL rows of one column in
//            registers and LPC neighbouring lanes share a column (D <= RPL * LPC); the two dot
//            products per token are reduced over those lanes with DPP swaps.  The rows of a chunk
//            of TB tokens (q, k, g, the block's v and b) are staged in LDS once per block; the next
//            chunk's rows are fetched into registers -- clamped loads, issued back to back -- before
//            the current chunk's dependent steps run; the chunk's outputs leave through LDS as
//            whole runs.  Steps with few (segment, head) pairs take the variant with more lanes per
//            column so that the grid still covers the chip.
//   single rows with D <= 256 and P a multiple of four go through state_step_kernel instead, which reads the state by rows.
//   gla and delta with D <= 256 take chunks of 16 tokens on the f32 matrix instructions instead (further down) in steps
//   with a segment of 32 rows or more, but for those that run_matrix_scan keeps here.
//
// mx_lru_scan: a diagonal recurrence per channel, S <- a S + sqrt(1 - a^2) i u with
//     a = exp(-8 sigmoid(zr + r_bias) softplus(lam)),  i = sigmoid(zi + i_bias),
//   output S * gelu_tanh(y + y_bias).  Two launches: the gates (a, the input term and the GeLU
//   branch: every transcendental; they replace z and u in place, in f32) elementwise over all rows,
//   then the recurrence itself, where a block of 16 channels walks 256 tokens at a time: each thread
//   scans 16 tokens of one channel from zero, the sixteen partial maps S -> A S + B are folded through
//   LDS, and the outputs are corrected by the true start state.  Steps of single rows (decode) take
//   one fused launch instead.  mx_lru_blocks has the block-diagonal product of zr and zi in the gates' launch as well.
//
// mx_mingru_scan: the minimal gated recurrent unit, S <- (1 - z) S + z c per channel with gates that read
//   only the current token: z = sigmoid(zp + z_bias), u = xp + x_bias, c = u + 1/2 for u >= 0 and
//   sigmoid(u) below; output S * silu(gp).  The same two launches (a gates pass that leaves 1 - z, z c
//   and the SiLU branch in f32, then the recurrence kernel above) or one fused launch for single rows.
#include <type_traits>

#include "mx_common.h"

namespace {

template <int LPC>
__device__ __forceinline__ float lane_group_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));      // quad_perm [1,0,3,2]
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));      // quad_perm [2,3,0,1]
  if (LPC >= 8) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));   // row_half_mirror
  if (LPC >= 16) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true));  // row_mirror
  return v;
}

__device__ __forceinline__ float ld_code(const void* p, int code, long i) {
  return code == 1 ? reinterpret_cast<const float*>(p)[i] : (float)reinterpret_cast<const bf16*>(p)[i];
}

// one block per token.  a [T, H*D] -> g in place; delta: aux[t] = [rq, rk per key/value head | b per head]
template <typename TQ, bool DELTA>
__global__ void scan_prep_kernel(const TQ* __restrict__ q, long sq, const TQ* __restrict__ k, long sk,
                                 float* __restrict__ a, long sa, const float* __restrict__ a_bias,
                                 const float* __restrict__ A_log, const void* __restrict__ beta, long sbeta,
                                 int beta_code, float tau_inv, float* __restrict__ aux, int H, int G, int D) {
  const long t = blockIdx.x;
  float* ar = a + t * sa;
  for (int e = threadIdx.x; e < H * D; e += blockDim.x) {
    const float z = ar[e] + a_bias[e];
    ar[e] = DELTA ? expf(-expf(A_log[e / D]) * mx_softplus(z)) : expf(-mx_softplus(-z) * tau_inv);
  }
  if (!DELTA) return;
  float* ax = aux + t * (2 * G + H);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const float qscale = 1.0f / sqrtf((float)D);
  for (int r = wave; r < 2 * G; r += nw) {          // row r: q head r / 2 or k head r / 2
    const TQ* src = (r & 1) ? k + t * sk + (r >> 1) * D : q + t * sq + (r >> 1) * D;
    float ss = 0.f;
    for (int d = lane; d < D; d += 64) {
      const float x = ldf(src + d);
      ss += x * x;
    }
    ss = mx_wave_sum(ss);
    if (lane == 0) ax[r] = ((r & 1) ? 1.0f : qscale) / sqrtf(ss + 1e-6f);
  }
  for (int h = threadIdx.x; h < H; h += blockDim.x) ax[2 * G + h] = mx_sigmoid(ld_code(beta, beta_code, t * sbeta + h));
}

// grid (ceil(P / CB), H, S), 256 threads = CB columns x LPC lanes, CB = 256 / LPC
// MODE 0: gla, 1: delta, 2: fixed decay per head (a_bias = decay [H], tau_inv = the output scale, beta_code =
// activation code | storage code of v << 4; q and k of type TQ, no g / aux / beta)
template <typename TQ, int RPL, int LPC, int MODE, bool ONE>      // ONE: every segment is a single row (decode)
__global__ void __launch_bounds__(256)
matrix_scan_kernel(const TQ* __restrict__ q, long sq, const TQ* __restrict__ k, long sk, const TQ* __restrict__ v, long sv,
                   const float* __restrict__ gdec, long sa, const float* __restrict__ aux, float* __restrict__ state,
                   const int* __restrict__ cu, const int* __restrict__ slot, const int* __restrict__ pos,
                   float* __restrict__ out, int H, int G, int D, int P, const float* __restrict__ a_bias,
                   const float* __restrict__ A_log, const void* __restrict__ beta, long sbeta, int beta_code,
                   float tau_inv, int most) {
  constexpr bool DELTA = MODE == 1, FIXED = MODE == 2;
  constexpr int DP = RPL * LPC;          // padded key size
  constexpr int CB = 256 / LPC;          // columns per block
  constexpr int TB = ONE ? 1 : (DP <= 256 ? 16 : 8);   // tokens per chunk
  constexpr int NE = (TB * DP + 255) / 256;            // staged (token, key channel) elements per thread
  constexpr int NV = (TB * CB + 255) / 256;
  __shared__ __align__(16) float qs[TB * DP];
  __shared__ __align__(16) float ks[TB * DP];
  __shared__ __align__(16) float gs[FIXED ? 4 : TB * DP];
  __shared__ float vs[TB * CB];
  __shared__ float os[TB * CB];
  __shared__ float bs[TB];
  const int s = blockIdx.z;
  const int sl = slot[s];
  if (sl < 0) return;
  const int r0 = cu[s], n = cu[s + 1] - r0;
  if (n <= 0 || n > most) return;        // longer ones are not this launch's
  const int h = blockIdx.y, kvh = h / (H / G);
  const int tid = threadIdx.x, part = tid % LPC, cl = tid / LPC;
  const int c0 = blockIdx.x * CB, col = c0 + cl;
  const bool fresh = pos[r0] == 0;
  const float qscale = 1.0f / sqrtf((float)D);
  const int AW = 2 * G + H;              // aux row width
  const float gfix = FIXED ? a_bias[h] : 1.f;
  const int fact = beta_code & 15, vcode = beta_code >> 4;

  float S[RPL];
  float* srec = state + (((long)sl * H + h) * D) * P;
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int d = part * RPL + i;
    S[i] = (!fresh && d < D && col < P) ? srec[(long)d * P + col] : 0.f;
  }

  // chunk rows in flight: element e = tid + 256 * i is (token e / DP, channel e % DP); loads are clamped
  // to the segment's last row and to channel D - 1, and masked when they land
  float pq[NE], pk[NE], pg[NE], pv[NV], pb = 0.f;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = min(tid + 256 * i, TB * DP - 1);
      const int t = e / DP, d = e - t * DP;
      const long row = r0 + min(t0 + t, n - 1);
      const int dc = min(d, D - 1);
      if (FIXED) {         // raw values: the activation waits until they are stored to LDS, so the loads stay in flight
        pq[i] = ldf(q + row * sq + kvh * D + dc);
        pk[i] = ldf(k + row * sk + kvh * D + dc);
      } else if (ONE) {       // no prep pass ran: the decay from its pre-activation here, the unit norms after staging
        pq[i] = ldf(q + row * sq + kvh * D + dc);
        pk[i] = ldf(k + row * sk + kvh * D + dc);
        const float z = gdec[row * sa + h * D + dc] + a_bias[h * D + dc];
        pg[i] = DELTA ? expf(-expf(A_log[h]) * mx_softplus(z)) : expf(-mx_softplus(-z) * tau_inv);
      } else {
        float rq = DELTA ? aux[row * AW + 2 * kvh] : 1.f, rk = DELTA ? aux[row * AW + 2 * kvh + 1] : 1.f;
        pq[i] = ldf(q + row * sq + kvh * D + dc) * rq;
        pk[i] = ldf(k + row * sk + kvh * D + dc) * rk;
        pg[i] = gdec[row * sa + h * D + dc];
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = min(tid + 256 * i, TB * CB - 1);
      const int t = e / CB, c = e - t * CB;
      const long vi = (long)(r0 + min(t0 + t, n - 1)) * sv + h * P + min(c0 + c, P - 1);
      if (FIXED) {
        pv[i] = ld_code(v, vcode, vi);
      } else {
        pv[i] = ldf(v + vi);
      }
    }
    if (DELTA && tid < TB)
      pb = ONE ? mx_sigmoid(ld_code(beta, beta_code, (long)(r0 + min(t0 + tid, n - 1)) * sbeta + h))
               : aux[(long)(r0 + min(t0 + tid, n - 1)) * AW + 2 * G + h];
  };
  fetch(0);
  for (int t0 = 0; t0 < n; t0 += TB) {
    const int nt = min(TB, n - t0);
    __syncthreads();                     // the previous chunk's outputs have left os; its rows are consumed
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = tid + 256 * i;
      if (e < TB * DP) {
        const bool live = (e % DP) < D;
        if (FIXED && fact == 1) {
          qs[e] = live ? mx_silu(pq[i]) : 0.f;
          ks[e] = live ? mx_silu(pk[i]) : 0.f;
        } else {
          qs[e] = live ? pq[i] : 0.f;
          ks[e] = live ? pk[i] : 0.f;
        }
        if (!FIXED) gs[e] = live ? pg[i] : 1.f;
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = tid + 256 * i;
      if (e < TB * CB) vs[e] = (c0 + e % CB) < P ? ((FIXED && fact == 1) ? mx_silu(pv[i]) : pv[i]) : 0.f;
    }
    if (DELTA && tid < TB) bs[tid] = pb;
    __syncthreads();
    if (ONE && DELTA) {                  // q (wave 0) and k (wave 1) become unit vectors
      const int wave = tid >> 6, lane = tid & 63;
      if (wave < 2) {
        float* buf = wave == 0 ? qs : ks;
        float ss = 0.f;
        for (int d = lane; d < DP; d += 64) ss += buf[d] * buf[d];
        ss = mx_wave_sum(ss);
        const float sc = (wave == 0 ? qscale : 1.0f) / sqrtf(ss + 1e-6f);
        for (int d = lane; d < DP; d += 64) buf[d] *= sc;
      }
      __syncthreads();
    }
    if (t0 + TB < n) fetch(t0 + TB);
    // ---- the recurrence
    for (int t = 0; t < nt; ++t) {
      const float4* kr = reinterpret_cast<const float4*>(ks + t * DP + part * RPL);
      const float4* gr = reinterpret_cast<const float4*>(gs + t * DP + part * RPL);
      const float4* qr = reinterpret_cast<const float4*>(qs + t * DP + part * RPL);
      float u = vs[t * CB + cl];
      float kreg[RPL];
#pragma unroll
      for (int i4 = 0; i4 < RPL / 4; ++i4) {
        const float4 kk = kr[i4];
        kreg[4 * i4] = kk.x; kreg[4 * i4 + 1] = kk.y; kreg[4 * i4 + 2] = kk.z; kreg[4 * i4 + 3] = kk.w;
      }
      if (DELTA) {
        float acc = 0.f;
#pragma unroll
        for (int i4 = 0; i4 < RPL / 4; ++i4) {
          const float4 gg = gr[i4];
          S[4 * i4] *= gg.x; S[4 * i4 + 1] *= gg.y; S[4 * i4 + 2] *= gg.z; S[4 * i4 + 3] *= gg.w;
          acc += S[4 * i4] * kreg[4 * i4] + S[4 * i4 + 1] * kreg[4 * i4 + 1] + S[4 * i4 + 2] * kreg[4 * i4 + 2] +
                 S[4 * i4 + 3] * kreg[4 * i4 + 3];
        }
        acc = lane_group_sum<LPC>(acc);
        u = bs[t] * (u - acc);
      }
      float o = 0.f;
#pragma unroll
      for (int i4 = 0; i4 < RPL / 4; ++i4) {
        const float4 qq = qr[i4];
        if (FIXED) {
          S[4 * i4] *= gfix; S[4 * i4 + 1] *= gfix; S[4 * i4 + 2] *= gfix; S[4 * i4 + 3] *= gfix;
        } else if (!DELTA) {
          const float4 gg = gr[i4];
          S[4 * i4] *= gg.x; S[4 * i4 + 1] *= gg.y; S[4 * i4 + 2] *= gg.z; S[4 * i4 + 3] *= gg.w;
        }
        S[4 * i4] += kreg[4 * i4] * u;
        S[4 * i4 + 1] += kreg[4 * i4 + 1] * u;
        S[4 * i4 + 2] += kreg[4 * i4 + 2] * u;
        S[4 * i4 + 3] += kreg[4 * i4 + 3] * u;
        o += S[4 * i4] * qq.x + S[4 * i4 + 1] * qq.y + S[4 * i4 + 2] * qq.z + S[4 * i4 + 3] * qq.w;
      }
      o = lane_group_sum<LPC>(o);
      if (part == 0) os[t * CB + cl] = DELTA ? o : o * (FIXED ? tau_inv : qscale);   // delta: the scale is part of q's norm factor
    }
    __syncthreads();
    for (int e = tid; e < nt * CB; e += 256) {
      const int t = e / CB, c = e - t * CB;
      if (c0 + c < P) out[(long)(r0 + t0 + t) * H * P + h * P + c0 + c] = os[e];
    }
  }
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int d = part * RPL + i;
    if (d < D && col < P) srec[(long)d * P + col] = S[i];
  }
}

__device__ __forceinline__ float gelu_tanh_f(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// elementwise over [T, R]: z[.., zr] <- a, z[.., zi] <- sqrt(1 - a^2) i u, then u <- gelu_tanh(y + y_bias)
// (f32: the branch is rounded once, with the product, not before it)
template <typename TY>
__global__ void lru_gates_kernel(float* __restrict__ u, float* __restrict__ z, int bsz, long T,
                                 const float* __restrict__ r_bias, const float* __restrict__ i_bias,
                                 const float* __restrict__ lam, const TY* __restrict__ y, long sy,
                                 const float* __restrict__ y_bias, int R) {
  const long total = T * R;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const long t = e / R;
    const int c = (int)(e - t * R);
    const int b = c / bsz, j = c - b * bsz;
    float* zp = z + ((long)b * T + t) * 2 * bsz + j;
    const float r = mx_sigmoid(zp[0] + r_bias[c]);
    const float i = mx_sigmoid(zp[bsz] + i_bias[c]);
    const float la = -8.0f * r * mx_softplus(lam[c]);             // log a
    zp[0] = expf(la);
    zp[bsz] = sqrtf(-expm1f(2.0f * la)) * i * u[e];               // 1 - a^2 without cancellation
    u[e] = gelu_tanh_f(ldf(y + t * sy + c) + (y_bias != nullptr ? y_bias[c] : 0.f));
  }
}

constexpr int LRU_CL = 16;      // tokens per thread
constexpr int LRU_NC = 16;      // thread chunks per block iteration
constexpr int LRU_CH = 16;      // channels per block (256 threads: 16 channels x 16 chunks, 256 tokens per iteration)

// grid (ceil(R / LRU_CH), S).  z holds a | input term, gy the GeLU branch (lru_gates_kernel).
template <typename TO>
__global__ void __launch_bounds__(256)
lru_scan_kernel(const float* __restrict__ z, const float* __restrict__ gy, int bsz, long T, float* __restrict__ state,
                const int* __restrict__ cu, const int* __restrict__ slot, const int* __restrict__ pos,
                TO* __restrict__ out, int R) {
  __shared__ float sA[LRU_NC][LRU_CH], sB[LRU_NC][LRU_CH], sS[LRU_CH];
  const int s = blockIdx.y;
  const int sl = slot[s];
  if (sl < 0) return;
  const int r0 = cu[s], n = cu[s + 1] - r0;
  if (n <= 0) return;
  const int ch = threadIdx.x % LRU_CH, j = threadIdx.x / LRU_CH;
  const int c = min((int)blockIdx.x * LRU_CH + ch, R - 1);
  const bool live = (int)blockIdx.x * LRU_CH + ch < R;
  const int b = c / bsz, jj = c - b * bsz;
  const float* zb = z + (long)b * T * 2 * bsz + jj;
  if (j == 0) sS[ch] = pos[r0] == 0 ? 0.f : state[(long)sl * R + c];
  for (int t0 = 0; t0 < n; t0 += LRU_CL * LRU_NC) {
    const int first = t0 + j * LRU_CL;
    const int cnt = max(0, min(LRU_CL, n - first));
    float A[LRU_CL], L[LRU_CL], Gy[LRU_CL];
    if (cnt > 0) {
#pragma unroll
      for (int i = 0; i < LRU_CL; ++i) {          // independent loads, issued together
        const long t = r0 + min(first + i, n - 1);
        A[i] = zb[t * 2 * bsz];
        L[i] = zb[t * 2 * bsz + bsz];
        Gy[i] = gy[t * R + c];
      }
    }
    float Pp = 1.f, Ll = 0.f;
#pragma unroll
    for (int i = 0; i < LRU_CL; ++i) {
      if (i < cnt) {
        Ll = A[i] * Ll + L[i];
        Pp *= A[i];
      }
      L[i] = Ll;      // state after token i from a zero start
      A[i] = Pp;      // product of the decays up to token i
    }
    sA[j][ch] = Pp;
    sB[j][ch] = Ll;
    __syncthreads();
    float S0 = sS[ch];
    for (int k = 0; k < j; ++k) S0 = sA[k][ch] * S0 + sB[k][ch];
#pragma unroll
    for (int i = 0; i < LRU_CL; ++i)
      if (i < cnt && live) stf(out + (long)(r0 + first + i) * R + c, (L[i] + A[i] * S0) * Gy[i]);
    __syncthreads();                             // every thread has read sS and the partial maps
    if (j == LRU_NC - 1) sS[ch] = Pp * S0 + Ll;
    __syncthreads();
  }
  if (j == 0 && live) state[(long)sl * R + c] = sS[ch];
}

// steps of single rows (decode): gates, recurrence and output in one launch, one thread per (row, channel)
template <typename TY, typename TO>
__global__ void lru_step_kernel(const float* __restrict__ u, const float* __restrict__ z, int bsz, long T,
                                const float* __restrict__ r_bias, const float* __restrict__ i_bias,
                                const float* __restrict__ lam, const TY* __restrict__ y, long sy,
                                const float* __restrict__ y_bias, float* __restrict__ state, const int* __restrict__ cu,
                                const int* __restrict__ slot, const int* __restrict__ pos, TO* __restrict__ out, int S,
                                int R) {
  const long total = (long)S * R;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int s = (int)(e / R), c = (int)(e - (long)s * R);
    const int sl = slot[s];
    const long t = cu[s];
    if (sl < 0 || cu[s + 1] <= t) continue;
    const int b = c / bsz, j = c - b * bsz;
    const float* zp = z + ((long)b * T + t) * 2 * bsz + j;
    const float r = mx_sigmoid(zp[0] + r_bias[c]);
    const float i = mx_sigmoid(zp[bsz] + i_bias[c]);
    const float la = -8.0f * r * mx_softplus(lam[c]);
    const float prev = pos[t] == 0 ? 0.f : state[(long)sl * R + c];
    const float Sn = expf(la) * prev + sqrtf(-expm1f(2.0f * la)) * i * u[t * R + c];
    state[(long)sl * R + c] = Sn;
    stf(out + t * R + c, Sn * gelu_tanh_f(ldf(y + t * sy + c) + (y_bias != nullptr ? y_bias[c] : 0.f)));
  }
}

__device__ __forceinline__ float mingru_candidate(float u) { return u >= 0.f ? u + 0.5f : mx_sigmoid(u); }

// elementwise over [T, R]: ab[t, c] <- 1 - z, ab[t, R + c] <- z * candidate, gy[t, c] <- silu(g), all f32
template <typename TI>
__global__ void mingru_gates_kernel(const TI* __restrict__ zp, long sz, const TI* __restrict__ xp, long sx,
                                    const TI* __restrict__ gp, long sg, const float* __restrict__ z_bias,
                                    const float* __restrict__ x_bias, float* __restrict__ ab, float* __restrict__ gy,
                                    long T, int R) {
  const long total = T * R;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const long t = e / R;
    const int c = (int)(e - t * R);
    const float a = ldf(zp + t * sz + c) + (z_bias != nullptr ? z_bias[c] : 0.f);
    const float u = ldf(xp + t * sx + c) + (x_bias != nullptr ? x_bias[c] : 0.f);
    ab[t * 2 * R + c] = mx_sigmoid(-a);                              // 1 - sigmoid(a) without cancellation
    ab[t * 2 * R + R + c] = mx_sigmoid(a) * mingru_candidate(u);
    gy[e] = mx_silu(ldf(gp + t * sg + c));
  }
}

// steps of single rows (decode): gates, recurrence and output in one launch, one thread per (row, channel)
template <typename TI, typename TO>
__global__ void mingru_step_kernel(const TI* __restrict__ zp, long sz, const TI* __restrict__ xp, long sx,
                                   const TI* __restrict__ gp, long sg, const float* __restrict__ z_bias,
                                   const float* __restrict__ x_bias, float* __restrict__ state,
                                   const int* __restrict__ cu, const int* __restrict__ slot, const int* __restrict__ pos,
                                   TO* __restrict__ out, int S, int R) {
  const long total = (long)S * R;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int s = (int)(e / R), c = (int)(e - (long)s * R);
    const int sl = slot[s];
    const long t = cu[s];
    if (sl < 0 || cu[s + 1] <= t) continue;
    const float a = ldf(zp + t * sz + c) + (z_bias != nullptr ? z_bias[c] : 0.f);
    const float u = ldf(xp + t * sx + c) + (x_bias != nullptr ? x_bias[c] : 0.f);
    const float prev = pos[t] == 0 ? 0.f : state[(long)sl * R + c];
    const float Sn = mx_sigmoid(-a) * prev + mx_sigmoid(a) * mingru_candidate(u);
    state[(long)sl * R + c] = Sn;
    stf(out + t * R + c, Sn * mx_silu(ldf(gp + t * sg + c)));
  }
}

// Single rows (decode): the token of matrix_scan_kernel's ONE form with the state read and written as it lies.  A block takes 32 of a head's
// value columns and all of its keys: eight lanes by four columns are 128 bytes of a row, 32 rows side by side, RPT of them a thread,
// all asked for before anything else.  The sums over the keys meet by lane exchanges and once through LDS.  Bound by the state's bytes and,
// for few rows, by latency.  16 heads, 15 rows, by columns (16-byte pieces of a row per lane group) / here, us: delta, 128 x 128 22.7 / 11.0, gla, 64 x
// 128 14.8 / 7.3; 8 heads, one row in f32 6.5 / 5.4 and 5.3 / 4.8.
template <typename TQ, int MODE, int RPT>
__global__ void __launch_bounds__(256)
state_step_kernel(const TQ* __restrict__ q, long sq, const TQ* __restrict__ k, long sk, const TQ* __restrict__ v, long sv,
                  const float* __restrict__ a, long sa, float* __restrict__ state, const int* __restrict__ cu, const int* __restrict__ slot,
                  const int* __restrict__ pos, float* __restrict__ out, int H, int G, int D, int P, const float* __restrict__ a_bias,
                  const float* __restrict__ A_log, const void* __restrict__ beta, long sbeta, int beta_code, float tau_inv, int most) {
  constexpr bool DELTA = MODE == 1, FIXED = MODE == 2;
  constexpr int DP = 32 * RPT;
  __shared__ float qs[DP], ks[DP], gs[DP], norm[2][4];
  __shared__ mx_f32x4 red[2][4][8];
  const int s = blockIdx.z, sl = slot[s];
  if (sl < 0) return;
  const long t = cu[s];
  const int n = cu[s + 1] - (int)t;
  if (n <= 0 || n > most) return;
  const int h = blockIdx.y, kvh = h / (H / G), tid = threadIdx.x, lane = tid & 63, w = tid >> 6, cg = tid & 7, rg = tid >> 3;
  const int c = blockIdx.x * 32 + 4 * cg, cc = min(c, P - 4);
  const bool fresh = pos[t] == 0;
  float* srec = state + (((long)sl * H + h) * D) * P + cc;
  mx_f32x4 S[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int d = 32 * i + rg;
    S[i] = !fresh && d < D ? ldf4_once(srec + (long)d * P) : mx_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  mx_f32x4 u;
  const int fact = beta_code & 15, vcode = beta_code >> 4;
  const long vi = t * sv + h * P + cc;
#pragma unroll
  for (int e = 0; e < 4; ++e) u[e] = FIXED ? ld_code(v, vcode, vi + e) : ldf(v + vi + e);
  float b = 1.f;
  if (DELTA) b = mx_sigmoid(ld_code(beta, beta_code, t * sbeta + h));
  const float qscale = 1.0f / sqrtf((float)D), gfix = FIXED ? a_bias[h] : 1.f;
  if (w < (DP + 63) / 64) {
    float qv = 0.f, kv = 0.f, gv = 1.f;
    if (tid < D) {
      qv = ldf(q + t * sq + kvh * D + tid);
      kv = ldf(k + t * sk + kvh * D + tid);
      if (!FIXED) {
        const float z = a[t * sa + h * D + tid] + a_bias[h * D + tid];
        gv = DELTA ? expf(-expf(A_log[h]) * mx_softplus(z)) : expf(-mx_softplus(-z) * tau_inv);
      }
      if (FIXED && fact == 1) qv = mx_silu(qv), kv = mx_silu(kv);
    }
    if (tid < DP) qs[tid] = qv, ks[tid] = kv, gs[tid] = gv;
    if (DELTA) {
      const float qq = mx_wave_sum(qv * qv), kk = mx_wave_sum(kv * kv);
      if (lane == 0) norm[0][w] = qq, norm[1][w] = kk;
    }
  }
  if (FIXED && fact == 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = mx_silu(u[e]);
  __syncthreads();
  float fq = 1.f, fk = 1.f;
  if (DELTA) {                             // q and k become unit vectors, q also scaled
    float qq = 0.f, kk = 0.f;
#pragma unroll
    for (int i = 0; i < (DP + 63) / 64; ++i) qq += norm[0][i], kk += norm[1][i];
    fq = qscale / sqrtf(qq + 1e-6f);
    fk = 1.0f / sqrtf(kk + 1e-6f);
  }
  auto total = [&](mx_f32x4 x, int at) {   // over all keys of this thread's columns
#pragma unroll
    for (int o = 8; o < 64; o <<= 1)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] += __shfl_xor(x[e], o, 64);
    if (lane < 8) red[at][w][lane] = x;
    __syncthreads();
    return (red[at][0][cg] + red[at][1][cg]) + (red[at][2][cg] + red[at][3][cg]);
  };
#pragma unroll
  for (int i = 0; i < RPT; ++i) S[i] *= FIXED ? gfix : gs[32 * i + rg];
  if (DELTA) {
    mx_f32x4 x = mx_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < RPT; ++i) x += S[i] * (ks[32 * i + rg] * fk);
    x = total(x, 0);
    u = b * (u - x);
  }
  mx_f32x4 o = mx_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int d = 32 * i + rg;
    S[i] += u * (ks[d] * fk);
    o += S[i] * (qs[d] * fq);
    if (d < D && c < P) stf4_once(srec + (long)d * P, S[i]);
  }
  o = total(o, 1);
  if (tid < 8 && c < P) stf4(out + t * H * P + h * P + c, DELTA ? o : o * (FIXED ? tau_inv : qscale));
}

template <typename TQ, int RPL, int LPC, int DELTA>
int launch_matrix_scan(const void* q, long sq, const void* k, long sk, const void* v, long sv, const float* g, long sa,
                       const float* aux, float* state, const int* cu, const int* slot, const int* pos, float* out, int S,
                       int H, int G, int D, int P, const float* a_bias, const float* A_log, const void* beta, long sbeta,
                       int beta_dt, float tau_inv, bool one, int most, hipStream_t st) {
  constexpr int CB = 256 / LPC;
  dim3 grid((P + CB - 1) / CB, H, S);
  if (one)
    matrix_scan_kernel<TQ, RPL, LPC, DELTA, true><<<grid, 256, 0, st>>>(
        (const TQ*)q, sq, (const TQ*)k, sk, (const TQ*)v, sv, g, sa, aux, state, cu, slot, pos, out, H, G, D, P, a_bias,
        A_log, beta, sbeta, beta_dt, tau_inv, most);
  else
    matrix_scan_kernel<TQ, RPL, LPC, DELTA, false><<<grid, 256, 0, st>>>(
        (const TQ*)q, sq, (const TQ*)k, sk, (const TQ*)v, sv, g, sa, aux, state, cu, slot, pos, out, H, G, D, P, a_bias,
        A_log, beta, sbeta, beta_dt, tau_inv, most);
  MX_RETURN_LAUNCH();
}

// the steps of single rows that state_step_kernel takes
template <typename TQ, int MODE>
int launch_state_step(bool& done, const void* q, long sq, const void* k, long sk, const void* v, long sv, const float* g, long sa, const float*,
                      float* state, const int* cu, const int* slot, const int* pos, float* out, int S, int H, int G, int D, int P,
                      const float* a_bias, const float* A_log, const void* beta, long sbeta, int beta_dt, float tau_inv, bool one, int most,
                      hipStream_t st) {
  done = one && D <= 256 && P % 4 == 0 && ((size_t)state | (size_t)out) % 16 == 0;
  if (!done) return 0;
  const dim3 grid((P + 31) / 32, H, S);
#define STATE_STEP(RPT)                                                                                                             \
  state_step_kernel<TQ, MODE, RPT><<<grid, 256, 0, st>>>((const TQ*)q, sq, (const TQ*)k, sk, (const TQ*)v, sv, g, sa, state, cu, slot, pos, \
                                                         out, H, G, D, P, a_bias, A_log, beta, sbeta, beta_dt, tau_inv, most)
  if (D <= 32) STATE_STEP(1);
  else if (D <= 64) STATE_STEP(2);
  else if (D <= 128) STATE_STEP(4);
  else STATE_STEP(8);
#undef STATE_STEP
  MX_RETURN_LAUNCH();
}

// the variant with 16 lanes per column when the narrow one would leave most of the chip idle
template <typename TQ, int DELTA, typename... Args>
int dispatch_matrix_scan(int D, bool wide, Args... args) {
  bool done;
  const int rc = launch_state_step<TQ, DELTA>(done, args...);
  if (done) return rc;
  if (D <= 32) return launch_matrix_scan<TQ, 8, 4, DELTA>(args...);
  if (D <= 64) return wide ? launch_matrix_scan<TQ, 4, 16, DELTA>(args...) : launch_matrix_scan<TQ, 16, 4, DELTA>(args...);
  if (D <= 128) return wide ? launch_matrix_scan<TQ, 8, 16, DELTA>(args...) : launch_matrix_scan<TQ, 32, 4, DELTA>(args...);
  if (D <= 256) return wide ? launch_matrix_scan<TQ, 16, 16, DELTA>(args...) : launch_matrix_scan<TQ, 32, 8, DELTA>(args...);
  return launch_matrix_scan<TQ, 32, 16, DELTA>(args...);
}

// ---- chunks of 16 tokens on the f32 matrix instructions (gla and delta, steps with longer segments).
// With G_t the product of a chunk's decays up to token t (per key channel), E_t that of the tokens behind t, and
// w(s, t) = G_t / G_s formed as the running product of the decays between them -- no quotients, no exponents of sums: every
// factor is the one that the token form applies, and none exceeds 1 --
//     A[t][s] = sum_d q_t k_s w(s, t)  (s <= t),   M[t][s] = sum_d k_t k_s w(s, t)  (s < t),
//     delta:  U = T V - W S,  T = (1 + b M)^-1 b,  W = T (k G)   by forward substitution;   gla:  U = V
//     O = (q G) S + A U,      S <- G_15 S + (k E)^T U.
// scan_chunk_prep_kernel makes A, T, W, q G, k E of all chunks at once, in the order of the matrix operands: 16 threads per
// s walk t with w in registers.  scan_chunk_kernel walks the chunks of a (segment, head, 16 value columns): the waves (four, eight for
// keys of 129 - 256) own equal parts of the key channels of S, in registers, the sums over channels meet in LDS, one barrier per chunk.
// Bound by the f32 matrix rate where many (segment, head) pairs run (3 D P products per token), by the chain of 26 dependent
// products per 16 tokens otherwise; the operands come three chunks ahead (one ahead: 144 against 125 us for the chain of 1500
// tokens).  16 heads, values of 128, token form -> both launches here: delta, D = 128, segments of 1500, 40, 600, 1 and 1
// tokens 509 -> 175 us (50 of them the preparation), four of 2048 865 -> 421, 64 + 40 + 32 tokens 41 -> 26; gla, D = 64,
// 279 -> 77, 433 -> 140 and 19 -> 16.  Errors against 64 bits are those of the token form.
typedef float f32x4 __attribute__((ext_vector_type(4)));

// The block-diagonal gates with their product: z[.., zr] = a, z[.., zi] = sqrt(1 - a^2) i u, gy = gelu_tanh(y + y_bias), by
// the functions of lru_gates_kernel: from equal sums the same bits.  A block takes 16 UT tokens and 64 channels of one part of bs, both of
// whose matrices (w [B][2 bs][bs], r over i) it stages with the tokens in three stages of 32 of K by LDS-DMA, 16-byte chunks swizzled by the row; a wave 16 channels, both
// gates in one lane, each sum in two halves.  Bound by the f32 products (46 us of the first figure) and the transcendentals.  R = 2048, 8 parts,
// with the library's product and lru_gates_kernel / here: 3453 rows 153 / 99, 1200 60 / 40, 100 25 / 8; operands straight from the caches,
// whose rows lie a power of two apart, 119.  Errors against 64 bits 1.9e-7 of the norm of a, of the library's product 2.9e-7.
template <typename TY, int UT>
__global__ void __launch_bounds__(256) lru_blocks_kernel(const float* __restrict__ u, const float* __restrict__ w, int bs, int T, int R,
                                                         const float* __restrict__ r_bias, const float* __restrict__ i_bias,
                                                         const float* __restrict__ lam, const TY* __restrict__ y, long sy,
                                                         const float* __restrict__ y_bias, float* __restrict__ z, float* __restrict__ gy) {
  constexpr int NST = 3, ROWS = 128 + 16 * UT, STG = ROWS * 128, PIECES = ROWS / 8, LPS = (PIECES + 3) / 4;
  __shared__ __attribute__((aligned(1024))) char smem[NST * STG];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const int cb = blockIdx.y * 64, b = cb / bs, jb = cb - b * bs, t0 = blockIdx.x * 16 * UT, n = bs / 32;
  const char* src[LPS];                            // of this lane in the wave's pieces of a stage: 64 rows for r, 64 for i, the tokens
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const int r = min(wv + 4 * i, PIECES - 1) * 8 + (lane >> 3), ch = (lane & 7) ^ ((r >> 1) & 7);
    const float* row = r < 128 ? w + ((long)b * 2 * bs + (r < 64 ? 0 : bs) + jb + (r & 63)) * bs : u + (long)min(t0 + r - 128, T - 1) * R + b * bs;
    src[i] = reinterpret_cast<const char*>(row + 4 * ch);
  }
  const unsigned lds0 = (unsigned)(uintptr_t)((__attribute__((address_space(3))) char*)smem);
  auto stage = [&](int t) {
#pragma unroll
    for (int i = 0; i < LPS; ++i) {
      unsigned keep;
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep)
                   : "v"(src[i] + 128 * t), "s"(lds0 + (t % NST) * STG + min(wv + 4 * i, PIECES - 1) * 1024)
                   : "memory");
    }
  };
  f32x4 acc[2][2][UT];                             // half of the sum, gate, token group
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int k = 0; k < UT; ++k) acc[h][d][k] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int at[2] = {(g ^ ((c >> 1) & 7)) << 4, ((4 + g) ^ ((c >> 1) & 7)) << 4};
  stage(0);
  if (n > 1) stage(1);
  for (int t = 0; t < n; ++t) {
    if (t + 1 < n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                  // stage t is there, and every wave has read stage t - 1
    if (t + 2 < n) stage(t + 2);
    const char* sm = smem + (t % NST) * STG + c * 128;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 p = *reinterpret_cast<const f32x4*>(sm + 16 * wv * 128 + at[h]);
      const f32x4 q = *reinterpret_cast<const f32x4*>(sm + (64 + 16 * wv) * 128 + at[h]);
      f32x4 x[UT];
#pragma unroll
      for (int k = 0; k < UT; ++k) x[k] = *reinterpret_cast<const f32x4*>(sm + (128 + 16 * k) * 128 + at[h]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int k = 0; k < UT; ++k) {
          acc[e & 1][0][k] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[k][e], p[e], acc[e & 1][0][k], 0, 0, 0);
          acc[e & 1][1][k] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[k][e], q[e], acc[e & 1][1][k], 0, 0, 0);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  const int ch = cb + 16 * wv + c, j = jb + 16 * wv + c;
  const float rb = r_bias[ch], ib = i_bias[ch], sp = -8.0f * mx_softplus(lam[ch]), yb = y_bias != nullptr ? y_bias[ch] : 0.f;
#pragma unroll
  for (int k = 0; k < UT; ++k)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = t0 + 16 * k + 4 * g + r;
      if (t >= T) continue;
      const float rr = mx_sigmoid(acc[0][0][k][r] + acc[1][0][k][r] + rb), ii = mx_sigmoid(acc[0][1][k][r] + acc[1][1][k][r] + ib);
      const float la = rr * sp;
      float* zp = z + ((long)b * T + t) * 2 * bs + j;
      zp[0] = expf(la);
      zp[bs] = sqrtf(-expm1f(2.0f * la)) * ii * u[(long)t * R + ch];
      gy[(long)t * R + ch] = gelu_tanh_f(ldf(y + t * sy + ch) + yb);
    }
}
constexpr int SCC = 16;                  // tokens per chunk
constexpr int SCAN_LEAST = 32;           // the longest segment from which the chunk form is taken (two chunks; see above)

__host__ __device__ inline long scan_chunk_floats(int DP, bool delta) { return 33L * DP + 256 + (delta ? 256 + 16L * DP : 0); }

// where (s, t) of A and T lies: wave s % 4 reads its 64 consecutive values
__device__ __forceinline__ int chunk_pair(int s, int t) { return (s & 3) * 64 + (s >> 2) * 16 + t; }

// exp(x) for x <= 0: the product with log2 e in two parts, so that the error is that of the exponential alone
__device__ __forceinline__ float exp_below(float x) {
  x = x < -150.f ? -150.f : x;
  const float h = x * 1.44269502f, l = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269502f, -h));
  const float e = __builtin_amdgcn_exp2f(h);
  return fmaf(e, l * 0.693147182f, e);
}

// exp(rate * softplus(z)), rate <= 0, without branches (the general functions took half of the chunk preparation's vector
// instructions: 8192 rows x 16 heads x 128 channels 200 -> 177 us).  log(1 + y) = 2 atanh(s), s = y / (2 + y) <= 1/3, by the
// series of atanh to s^17, whose rest is below 2^-29 of the sum.
__device__ __forceinline__ float decay_of(float z, float rate) {
  const float y = exp_below(-fabsf(z)), d = 2.f + y;
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.f), r, r);
  const float s = y * r, q = s * s;
  float p = 1.f / 17;
  p = fmaf(p, q, 1.f / 15);
  p = fmaf(p, q, 1.f / 13);
  p = fmaf(p, q, 1.f / 11);
  p = fmaf(p, q, 1.f / 9);
  p = fmaf(p, q, 1.f / 7);
  p = fmaf(p, q, 1.f / 5);
  p = fmaf(p, q, 1.f / 3);
  const float s2 = 2.f * s, sp = (z < 0.f ? 0.f : z) + fmaf(s2 * q, p, s2);
  return exp_below(rate * sp);
}

// grid (T / 16 + S, H): chunk x of the step; segment s starts at chunk cu[s] / 16 + s
template <typename TQ, int DP, bool DELTA>
__global__ void __launch_bounds__(256, 2)
scan_chunk_prep_kernel(const TQ* __restrict__ q, long sq, const TQ* __restrict__ k, long sk, const float* __restrict__ a,
                       long sa, const float* __restrict__ a_bias, const float* __restrict__ A_log,
                       const void* __restrict__ beta, long sbeta, int beta_code, float tau_inv, float* __restrict__ ws,
                       const int* __restrict__ cu, const int* __restrict__ slot, int S, int H, int G, int D, int least) {
  constexpr int LD = DP + 4;             // 16 rows at one column meet different banks
  __shared__ __align__(16) float qs[SCC * LD], ks[SCC * LD], gs[SCC * LD];
  __shared__ __align__(16) float As[SCC * SCC], Ms[SCC * SCC];
  __shared__ float bs[SCC];
  const int h = blockIdx.y, kvh = h / (H / G), tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ci = blockIdx.x;
  int s = 0;
  for (int lo = 0, hi = S; lo < hi;) {   // the last segment that starts at or before this chunk
    const int mid = (lo + hi) >> 1;
    if (cu[mid] / SCC + mid <= ci) {
      s = mid;
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  const int first = (ci - cu[s] / SCC - s) * SCC, n = cu[s + 1] - cu[s];
  if (slot[s] < 0 || n < (DELTA ? least : 1) || first < 0 || first >= n) return;
  const long row0 = cu[s] + first;
  const int nt = min(SCC, n - first);
  const float qscale = 1.0f / sqrtf((float)D);
  const float rate = DELTA ? -expf(A_log[h]) : -tau_inv;
  constexpr int NE = SCC * DP / 256;     // elements per thread, in rows of its wave; loads are clamped and issued together
  const int d0 = tid % DP, dc = min(d0, D - 1), tw = wave * 64 / DP;
  TQ xq[NE], xk[NE];
  float xa[NE];
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const long row = row0 + min(tw + i * (256 / DP), nt - 1);
    xq[i] = (q + row * sq + kvh * D)[dc];
    xk[i] = (k + row * sk + kvh * D)[dc];
    xa[i] = (a + row * sa + h * D)[dc];
  }
  const float xb = a_bias[h * D + dc];
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int t = tw + i * (256 / DP);
    const bool live = t < nt && d0 < D;
    const float z = xa[i] + xb;
    qs[t * LD + d0] = live ? ldf(&xq[i]) * (DELTA ? 1.f : qscale) : 0.f;
    ks[t * LD + d0] = live ? ldf(&xk[i]) : 0.f;
    gs[t * LD + d0] = live ? decay_of(DELTA ? z : -z, rate) : 1.f;
  }
  As[tid] = Ms[tid] = 0.f;
  if (DELTA && tid < SCC) bs[tid] = tid < nt ? mx_sigmoid(ld_code(beta, beta_code, (row0 + tid) * sbeta + h)) : 0.f;
  __syncthreads();
  if (DELTA) {                           // unit rows of q (scaled) and k
    for (int r = wave; r < 2 * SCC; r += 4) {
      float* x = (r & 1 ? ks : qs) + (r >> 1) * LD;
      float ss = 0.f;
      for (int d = lane; d < DP; d += 64) ss += x[d] * x[d];
      ss = mx_wave_sum(ss);
      const float f = ((r & 1) ? 1.0f : qscale) / sqrtf(ss + 1e-6f);
      for (int d = lane; d < DP; d += 64) x[d] *= f;
    }
    __syncthreads();
  }
  {                                      // 16 lanes share s: channels 4 dg .. + 3 of every 64
    const int sj = tid >> 4, dg = (tid & 15) * 4;
    f32x4 w[DP / 64];
#pragma unroll
    for (int j = 0; j < DP / 64; ++j) w[j] = *reinterpret_cast<const f32x4*>(ks + sj * LD + 64 * j + dg);
    auto row = [&](int t, auto edge) {   // edge: some of this wave's s lie at or behind t
      float aq = 0.f, ak = 0.f;
#pragma unroll
      for (int j = 0; j < DP / 64; ++j) {
        const f32x4 qq = *reinterpret_cast<const f32x4*>(qs + t * LD + 64 * j + dg);
        const f32x4 gg = *reinterpret_cast<const f32x4*>(gs + t * LD + 64 * j + dg);
        if (!edge.value || t > sj) w[j] *= gg;
        aq += qq[0] * w[j][0] + qq[1] * w[j][1] + qq[2] * w[j][2] + qq[3] * w[j][3];
        if (DELTA) {
          const f32x4 kk = *reinterpret_cast<const f32x4*>(ks + t * LD + 64 * j + dg);
          ak += kk[0] * w[j][0] + kk[1] * w[j][1] + kk[2] * w[j][2] + kk[3] * w[j][3];
        }
      }
      aq = lane_group_sum<16>(aq);
      if (DELTA) ak = lane_group_sum<16>(ak);
      if (dg == 0 && t >= sj) {
        As[chunk_pair(sj, t)] = aq;
        if (DELTA && t > sj) Ms[t * SCC + sj] = ak;
      }
    };
#pragma unroll
    for (int t = 0; t < 4; ++t) row(4 * wave + t, std::true_type{});
    for (int t = 4 * wave + 4; t < SCC; ++t) row(t, std::false_type{});
  }
  __syncthreads();
  float* out = ws + ((long)ci * H + h) * scan_chunk_floats(DP, DELTA);
  for (int d = tid; d < DP + (DELTA ? SCC : 0); d += 256) {
    float x[SCC], g = 1.f;
#pragma unroll
    for (int t = 0; t < SCC; ++t) {
      float r;
      if (d < DP) {
        g *= gs[t * LD + d];
        qs[t * LD + d] *= g;
        r = ks[t * LD + d] * g;
      } else {
        r = t == d - DP ? 1.f : 0.f;
      }
      if (DELTA) {
#pragma unroll
        for (int i = 0; i < t; ++i) r -= Ms[t * SCC + i] * x[i];
        x[t] = r * bs[t];
      }
    }
    if (d < DP) {
      out[32 * DP + d] = g;
      float e = 1.f;
#pragma unroll
      for (int t = SCC - 1; t >= 0; --t) {
        const float gt = gs[t * LD + d];
        ks[t * LD + d] *= e;
        e *= gt;
        if (DELTA) gs[t * LD + d] = -x[t];
      }
    } else if (DELTA) {
#pragma unroll
      for (int t = 0; t < SCC; ++t) out[33 * DP + 256 + chunk_pair(d - DP, t)] = x[t];
    }
  }
  __syncthreads();
  out[33 * DP + tid] = As[tid];
  for (int e = tid; e < 4 * DP; e += 256) {                      // 16-byte operand pieces: tile e / 64, lane e % 64
    const int j = (e >> 6) * 16, c = e & 15, g = (e >> 4) & 3;
    *reinterpret_cast<f32x4*>(out + 4 * e) = *reinterpret_cast<const f32x4*>(qs + c * LD + j + 4 * g);
    f32x4 x;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = ks[(4 * g + r) * LD + j + c];
    *reinterpret_cast<f32x4*>(out + 16 * DP + 4 * e) = x;
    if (DELTA)
      *reinterpret_cast<f32x4*>(out + 33 * DP + 512 + 4 * e) = *reinterpret_cast<const f32x4*>(gs + c * LD + j + 4 * g);
  }
}

// grid (H, ceil(P / 16), S): all column blocks of a head on one chiplet, whose cache then holds the chunk's operands
template <typename TQ, int DP, int NW, bool DELTA>
__global__ void __launch_bounds__(NW * 64, 2)
scan_chunk_kernel(const TQ* __restrict__ v, long sv, const float* __restrict__ ws, float* __restrict__ state,
                  const int* __restrict__ cu, const int* __restrict__ slot, const int* __restrict__ pos,
                  float* __restrict__ out, int H, int D, int P, int least) {
  constexpr int TPW = DP / 16 / NW;      // tiles of 16 key channels per wave
  __shared__ __align__(16) f32x4 us[2][NW][64];
  __shared__ __align__(16) f32x4 os[2][NW][64];
  const int h = blockIdx.x, s = blockIdx.z;
  const int sl = slot[s], r0 = cu[s], n = cu[s + 1] - r0;
  if (sl < 0 || n < (DELTA ? least : 1)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c = lane & 15;
  const int col = blockIdx.y * 16 + c;
  const bool cok = col < P;
  float* srec = state + ((long)sl * H + h) * D * P;
  f32x4 S[TPW];
  const bool fresh = pos[r0] == 0;
#pragma unroll
  for (int j = 0; j < TPW; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * (w * TPW + j) + 4 * g + r;
      S[j][r] = !fresh && cok && d < D ? srec[(long)d * P + col] : 0.f;
    }
  const long step = (long)H * scan_chunk_floats(DP, DELTA);
  const float* base = ws + (long)(r0 / SCC + s) * step + h * scan_chunk_floats(DP, DELTA);
  const int last = (n - 1) / SCC;
  struct Chunk {
    f32x4 q[TPW], k[TPW], w[TPW], g[TPW];
    TQ v[4];
    float a, t;
  };
  const TQ* vp = v + (long)r0 * sv + h * P + min(col, P - 1);
  const TQ* vf = vp + 4 * g * sv;
  auto fetch = [&](Chunk& x, int t0) {   // x: the chunk of tokens t0 .. (behind the end: the last one again)
    const float* p = base + min(t0 / SCC, last) * step;
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      const int o = ((w * TPW + j) * 64 + lane) * 4;
      x.q[j] = *reinterpret_cast<const f32x4*>(p + o);
      x.k[j] = *reinterpret_cast<const f32x4*>(p + 16 * DP + o);
      if (DELTA) x.w[j] = *reinterpret_cast<const f32x4*>(p + 33 * DP + 512 + o);
      x.g[j] = *reinterpret_cast<const f32x4*>(p + 32 * DP + 16 * (w * TPW + j) + 4 * g);
    }
    x.a = p[33 * DP + (tid & 255)];
    if (DELTA) x.t = p[33 * DP + 256 + (tid & 255)];
    if (t0 + SCC <= n) {                 // (64-bit products are slow: only the tail forms them)
#pragma unroll
      for (int r = 0; r < 4; ++r) x.v[r] = vf[r * sv];
      vf += SCC * sv;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) x.v[r] = vp[min(t0 + 4 * g + r, n - 1) * sv];
    }
  };
  auto mine = [&](const f32x4& x) {      // tokens 4 g + w of a tile: this wave's K step (the first four waves')
    const float y = w == 0 ? x[0] : w == 1 ? x[1] : w == 2 ? x[2] : x[3];
    return NW == 4 || w < 4 ? y : 0.f;
  };
  float* op = out + (long)(r0 + 4 * g + w) * H * P + h * P + col;
  const long orow = (long)SCC * H * P;
  auto flush = [&](int t0, int buf) {    // a finished chunk: this wave's rows 4 g + w (the first four waves)
    const int t = t0 + 4 * g + w;
    const float* o = reinterpret_cast<const float*>(&os[buf][0][0]) + lane * 4 + (w & 3);
    float y = (o[0] + o[256]) + (o[512] + o[768]);
    if (NW == 8) y += (o[1024] + o[1280]) + (o[1536] + o[1792]);
    if (t < n && cok && w < 4) *op = y;
    op += orow;
  };
  auto walk = [&](Chunk& cur, Chunk& nxt, int t0, int buf) {
    fetch(nxt, t0 + 3 * SCC);
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 u, o[2] = {zero, zero};
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = t0 + 4 * g + r < n && cok ? ldf(&cur.v[r]) : 0.f;
    int bad = mx_drop_nonfinite(u, g);
    if (DELTA) {
      // two sums: the many small terms of W S are not rounded at the size of T V
      f32x4 x[2] = {zero, zero};
      const f32x4 tv = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.t, mine(u), zero, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < TPW; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.w[j][r], S[j][r], x[j & 1], 0, 0, 0);
      x[0] += TPW > 1 ? x[1] + tv : tv;
      us[buf][w][lane] = x[0];
    }
#pragma unroll
    for (int j = 0; j < TPW; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.q[j][r], S[j][r], o[j & 1], 0, 0, 0);
    if (TPW > 1) o[0] += o[1];
    __syncthreads();
    if (DELTA) {
      u = (us[buf][0][lane] + us[buf][1][lane]) + (us[buf][2][lane] + us[buf][3][lane]);
      if (NW == 8) u += (us[buf][NW - 4][lane] + us[buf][NW - 3][lane]) + (us[buf][NW - 2][lane] + us[buf][NW - 1][lane]);
      bad = min(bad, mx_drop_nonfinite(u, g));
    }
    if (t0 > 0) flush(t0 - SCC, buf ^ 1);
    o[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.a, mine(u), o[0], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      S[j] *= cur.g[j];
#pragma unroll
      for (int r = 0; r < 4; ++r) S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.k[j][r], u[r], S[j], 0, 0, 0);
    }
    if (bad < SCC) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[0][r] = 4 * g + r >= bad ? NAN : o[0][r];
#pragma unroll
      for (int j = 0; j < TPW; ++j) S[j] = f32x4{NAN, NAN, NAN, NAN};
    }
    os[buf][w][lane] = o[0];
  };
  // three chunks ahead: a chunk's step is shorter than the way to memory
  Chunk x[4];
#pragma unroll
  for (int i = 0; i < 3; ++i) fetch(x[i], i * SCC);
  for (int t0 = 0; t0 < n; t0 += 4 * SCC) {
    walk(x[0], x[3], t0, 0);
    if (t0 + SCC >= n) break;
    walk(x[1], x[0], t0 + SCC, 1);
    if (t0 + 2 * SCC >= n) break;
    walk(x[2], x[1], t0 + 2 * SCC, 0);
    if (t0 + 3 * SCC >= n) break;
    walk(x[3], x[2], t0 + 3 * SCC, 1);
  }
  __syncthreads();
  flush(last * SCC, last & 1);
#pragma unroll
  for (int j = 0; j < TPW; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * (w * TPW + j) + 4 * g + r;
      if (cok && d < D) srec[(long)d * P + col] = S[j][r];
    }
}

template <typename TQ, int TPW, bool DELTA>
int launch_scan_chunks(const void* q, long sq, const void* k, long sk, const void* v, long sv, const float* a, long sa,
                       const float* a_bias, const float* A_log, const void* beta, long sbeta, int beta_dt, float tau_inv,
                       float* ws, float* state, const int* cu, const int* slot, const int* pos, float* out, int S, int T,
                       int H, int G, int D, int P, int least, hipStream_t st) {
  scan_chunk_prep_kernel<TQ, 64 * TPW, DELTA><<<dim3(T / SCC + S, H), 256, 0, st>>>(
      (const TQ*)q, sq, (const TQ*)k, sk, a, sa, a_bias, A_log, beta, sbeta, beta_dt, tau_inv, ws, cu, slot, S, H, G, D, least);
  constexpr int NW = TPW <= 2 ? 4 : 8;
  scan_chunk_kernel<TQ, 64 * TPW, NW, DELTA><<<dim3(H, (P + 15) / 16, S), NW * 64, 0, st>>>((const TQ*)v, sv, ws, state, cu, slot,
                                                                                          pos, out, H, D, P, least);
  MX_RETURN_LAUNCH();
}

template <typename TQ, bool DELTA>
int run_matrix_scan(const void* q, long sq, const void* k, long sk, const void* v, long sv, float* a, long sa,
                    const float* a_bias, const float* A_log, const void* beta, long sbeta, int beta_dt, float tau_inv,
                    float* aux, float* ws, float* state, const int* cu, const int* slot, const int* pos, float* out, int S,
                    int T, int H, int G, int D, int P, int max_len, hipStream_t st) {
  // Steps of segments that are short on average are decode rows beside a prompt or two.  In the delta form a single row takes a
  // chunk as long as 16 do, and the single-row form a quarter of that: with more than 256 blocks' worth of rows the single ones
  // go there (16 heads of 128 x 128, us, all in chunks / apart / token form: 64 single rows beside 32 rows 96 / 50 / 92, 16 beside
  // 128 41 / 38 / 64; with longer prompts the rows hide behind the chain: 32 beside 1000 119 / 124 / 340), and steps below that
  // of at most two full chunks stay in the token form (8 heads, 21 beside three of 32 33 / 37 / 28).  Gla's chunks are cheaper.
  const bool rows = DELTA && T < 32L * S;
  const bool split = rows && max_len >= SCAN_LEAST && max_len <= 256 && (long)S * H * P > 256L * 128 && ws != nullptr && D <= 256;
  // the longest segment sets the step's duration: count the segments that can be about that long (a
  // prompt chunk beside many single decode rows is still one long chain)
  const long seff = max_len > 0 && !split ? (S < (T + max_len - 1) / max_len ? S : (T + max_len - 1) / max_len) : S;
  // Keys pad to 64 or 128 channels in chunks and not in the token form.  Where its blocks of 64 value columns fill the chip its
  // chains no longer matter, and it is the faster form (us, token / chunks of 32 segments of 100 tokens, 64 heads with values of
  // 64: delta, keys of 16 134 / 319, 64 240 / 341, 128 517 / 521; gla, 32 100 / 142, 64 183 / 126; 16 segments of 40, 32 heads,
  // delta, 64: 45 / 54).
  const long blocks64 = seff * H * ((P + 63) / 64);
  const bool brief = max_len < 64;
  long full = 1L << 62;
  if (D <= 32) full = DELTA || brief ? 256 : 512;
  else if (DELTA && D <= 96) full = brief ? 256 : D <= 64 ? 512 : 1024;
  const bool chunks = split || (ws != nullptr && max_len >= SCAN_LEAST && D <= 256 && !(rows && S >= 16 && max_len < 48) &&
                                blocks64 < full);
  if (chunks) {
    const int least = split ? 2 : 1;
#define SCAN_CHUNKS(TPW)                                                                                                  \
  launch_scan_chunks<TQ, TPW, DELTA>(q, sq, k, sk, v, sv, a, sa, a_bias, A_log, beta, sbeta, beta_dt, tau_inv, ws, state, \
                                     cu, slot, pos, out, S, T, H, G, D, P, least, st)
    const int rc = D <= 64 ? SCAN_CHUNKS(1) : D <= 128 ? SCAN_CHUNKS(2) : SCAN_CHUNKS(4);
#undef SCAN_CHUNKS
    if (rc || !split) return rc;
  }
  const bool one = max_len == 1 || split;          // single rows: no chunk staging
  if (!one)        // single-row steps fold this pass into the scan (one launch less per layer)
    scan_prep_kernel<TQ, DELTA><<<T, 256, 0, st>>>((const TQ*)q, sq, (const TQ*)k, sk, a, sa, a_bias, A_log, beta, sbeta,
                                                   beta_dt, tau_inv, aux, H, G, D);
  const int lpc = D <= 128 ? 4 : (D <= 256 ? 8 : 16);
  const long blocks = seff * H * ((P + 256 / lpc - 1) / (256 / lpc));
  return dispatch_matrix_scan<TQ, DELTA>(D, blocks < 512, q, sq, k, sk, v, sv, (const float*)a, sa, (const float*)aux, state,
                                         cu, slot, pos, out, S, H, G, D, P, a_bias, A_log, beta, sbeta, beta_dt, tau_inv,
                                         one, split ? 1 : 0x7fffffff, st);
}

}  // namespace

// q, k [rows, G*D] and v [rows, H*P] slices of storage type dt (row strides sq, sk, sv); a f32 [T, H*D]
// slice (row stride sa), which the token form of longer segments overwrites with the decays; a_bias f32 [H*D]; delta != 0: A_log f32 [H], beta
// [T, >= H] slice of type beta_dt, aux f32 [T, 2*G + H] scratch of that form; state f32 [slots, H, D, P]; out f32
// [T, H*P].  T: rows of the step (every row belongs to a segment or is padding); max_len: the longest
// segment (1: the decode form).  ws: f32 scratch of
// (T / 16 + S) * H * scan_chunk_floats(D padded to 64, 128 or 256) values for the chunk form, or null (token form).
MX_API int mx_matrix_scan(const void* q, long sq, const void* k, long sk, const void* v, long sv, int dt, float* a,
                          long sa, const float* a_bias, const float* A_log, const void* beta, long sbeta, int beta_dt,
                          float tau, int delta, float* aux, float* ws, float* state, const int* cu, const int* slot,
                          const int* pos, float* out, int S, int T, int max_len, int H, int G, int D, int P, hipStream_t st) {
  if (S <= 0 || T <= 0) return 0;
  if (D < 1 || D > 512 || G < 1 || H % G || tau <= 0.f || (delta && (A_log == nullptr || beta == nullptr || aux == nullptr)))
    return (int)hipErrorInvalidValue;
  const float ti = 1.0f / tau;
  if (delta) {
    if (dt == 1)
      return run_matrix_scan<float, true>(q, sq, k, sk, v, sv, a, sa, a_bias, A_log, beta, sbeta, beta_dt, ti, aux, ws, state,
                                          cu, slot, pos, out, S, T, H, G, D, P, max_len, st);
    return run_matrix_scan<bf16, true>(q, sq, k, sk, v, sv, a, sa, a_bias, A_log, beta, sbeta, beta_dt, ti, aux, ws, state, cu,
                                       slot, pos, out, S, T, H, G, D, P, max_len, st);
  }
  if (dt == 1)
    return run_matrix_scan<float, false>(q, sq, k, sk, v, sv, a, sa, a_bias, A_log, beta, sbeta, beta_dt, ti, aux, ws, state,
                                         cu, slot, pos, out, S, T, H, G, D, P, max_len, st);
  return run_matrix_scan<bf16, false>(q, sq, k, sk, v, sv, a, sa, a_bias, A_log, beta, sbeta, beta_dt, ti, aux, ws, state, cu,
                                      slot, pos, out, S, T, H, G, D, P, max_len, st);
}

// One fixed decay per head: S <- decay[h] S + act(k) act(v)^T, o = S^T act(q) * out_scale.  q, k [rows, H*D]
// slices of storage type dt_qk, v [rows, H*P] slice of type dt_v (the two may differ: rotated f32 q, k beside
// the projection's own v); act 0: none, 1: SiLU on q, k and v; decay f32 [H]; state f32 [slots, H, D, P];
// out f32 [T, H*P].  One launch, also for prompt chunks.
MX_API int mx_decay_scan(const void* q, long sq, const void* k, long sk, int dt_qk, const void* v, long sv, int dt_v,
                         int act, const float* decay, float out_scale, float* state, const int* cu, const int* slot,
                         const int* pos, float* out, int S, int T, int max_len, int H, int D, int P, hipStream_t st) {
  if (S <= 0 || T <= 0) return 0;
  if (D < 1 || D > 512 || decay == nullptr || (act != 0 && act != 1)) return (int)hipErrorInvalidValue;
  const bool one = max_len == 1;
  const long seff = max_len > 0 ? (S < (T + max_len - 1) / max_len ? S : (T + max_len - 1) / max_len) : S;
  const int lpc = D <= 128 ? 4 : (D <= 256 ? 8 : 16);
  const long blocks = seff * H * ((P + 256 / lpc - 1) / (256 / lpc));
  const int code = act | (dt_v << 4);
  // v travels as an untyped pointer: the fixed mode reads it by its storage code
  if (dt_qk == 1)
    return dispatch_matrix_scan<float, 2>(D, blocks < 512, q, sq, k, sk, v, sv, (const float*)nullptr, 0L,
                                          (const float*)nullptr, state, cu, slot, pos, out, S, H, H, D, P, decay,
                                          (const float*)nullptr, (const void*)nullptr, 0L, code, out_scale, one, 0x7fffffff, st);
  return dispatch_matrix_scan<bf16, 2>(D, blocks < 512, q, sq, k, sk, v, sv, (const float*)nullptr, 0L,
                                       (const float*)nullptr, state, cu, slot, pos, out, S, H, H, D, P, decay,
                                       (const float*)nullptr, (const void*)nullptr, 0L, code, out_scale, one, 0x7fffffff, st);
}

// u f32 [T, R], OVERWRITTEN with the GeLU branch; z f32 [blocks, T, 2 * R / blocks], OVERWRITTEN with the gates; y [T, >= R] slice (row stride
// sy, type dt_y); state f32 [slots, R]; out [T, R] of type dt_out
MX_API int mx_lru_scan(float* u, float* z, int blocks, const float* r_bias, const float* i_bias,
                       const float* lam, const void* y, long sy, int dt_y, const float* y_bias, float* state,
                       const int* cu, const int* slot, const int* pos, void* out, int dt_out, int S, int R, int T,
                       int max_len, hipStream_t st) {
  if (S <= 0 || T <= 0) return 0;
  if (blocks < 1 || R % blocks) return (int)hipErrorInvalidValue;
  if (max_len == 1) {
    const long tot = (long)S * R;
    const int g1 = (int)((tot + 255) / 256 < 8192 ? (tot + 255) / 256 : 8192);
    MX_DISPATCH(dt_y, TY, MX_DISPATCH(dt_out, TO, lru_step_kernel<TY, TO><<<g1, 256, 0, st>>>(
        u, z, R / blocks, (long)T, r_bias, i_bias, lam, (const TY*)y, sy, y_bias, state, cu, slot, pos, (TO*)out, S, R)));
    MX_RETURN_LAUNCH();
  }
  const long total = (long)T * R;
  const int gb = (int)((total + 255) / 256 < 8192 ? (total + 255) / 256 : 8192);
  MX_DISPATCH(dt_y, TY, lru_gates_kernel<TY><<<gb, 256, 0, st>>>(u, z, R / blocks, (long)T, r_bias, i_bias, lam, (const TY*)y,
                                                                 sy, y_bias, R));
  dim3 grid((R + LRU_CH - 1) / LRU_CH, S);
  MX_DISPATCH(dt_out, TO, lru_scan_kernel<TO><<<grid, 256, 0, st>>>(z, u, R / blocks, (long)T, state, cu, slot, pos, (TO*)out, R));
  MX_RETURN_LAUNCH();
}

// mx_lru_scan from the parts' matrices w f32 [blocks][2 R / blocks][R / blocks] (r over i): u f32 [T, R] is only read, z f32 [blocks, T,
// 2 R / blocks] and gy f32 [T, R] are scratch.  R / blocks in whole 64s, T R below 2^31, 16-byte operands.
MX_API int mx_lru_blocks(const float* u, const float* w, int blocks, const float* r_bias, const float* i_bias, const float* lam,
                         const void* y, long sy, int dt_y, const float* y_bias, float* z, float* gy, float* state, const int* cu,
                         const int* slot, const int* pos, void* out, int dt_out, int S, int R, int T, hipStream_t st) {
  if (S <= 0 || T <= 0) return 0;
  if (blocks < 1 || R < 1 || R % blocks || R / blocks % 64 || R / 64 > 65535 || S > 65535 || (long)T * R >= 1L << 31 ||
      ((size_t)u | (size_t)w) % 16)
    return (int)hipErrorInvalidValue;
  const int bs = R / blocks;
  // tokens per block: the fewest that leave more blocks than fit at once, 16 where the chip is not filled
  const long parts = R / 64;
  const int ut = (T + 63) / 64 * parts >= 1024 ? 4 : (T + 31) / 32 * parts >= 256 ? 2 : 1;
  const dim3 gg((T + 16 * ut - 1) / (16 * ut), (unsigned)parts);
#define LRU_BLOCKS(UT) \
  MX_DISPATCH(dt_y, TY, lru_blocks_kernel<TY, UT><<<gg, 256, 0, st>>>(u, w, bs, T, R, r_bias, i_bias, lam, (const TY*)y, sy, y_bias, z, gy))
  if (ut == 4) LRU_BLOCKS(4);
  else if (ut == 2) LRU_BLOCKS(2);
  else LRU_BLOCKS(1);
#undef LRU_BLOCKS
  const int rc = (int)hipGetLastError();
  if (rc) return rc;
  dim3 grid((R + LRU_CH - 1) / LRU_CH, S);
  MX_DISPATCH(dt_out, TO, lru_scan_kernel<TO><<<grid, 256, 0, st>>>(z, gy, bs, (long)T, state, cu, slot, pos, (TO*)out, R));
  MX_RETURN_LAUNCH();
}

// zp, xp, gp [T, >= R] slices of type dt_in (row strides sz, sx, sg): pre-activations of the update gate, of
// the candidate and of the output gate; z_bias, x_bias f32 [R] or null; ab f32 [T, 2R] and gy f32 [T, R]:
// scratch (unused by single-row steps); state f32 [slots, R]; out [T, R] of type dt_out
MX_API int mx_mingru_scan(const void* zp, long sz, const void* xp, long sx, const void* gp, long sg, int dt_in,
                          const float* z_bias, const float* x_bias, float* ab, float* gy, float* state, const int* cu,
                          const int* slot, const int* pos, void* out, int dt_out, int S, int R, int T, int max_len,
                          hipStream_t st) {
  if (S <= 0 || T <= 0) return 0;
  if (R < 1) return (int)hipErrorInvalidValue;
  if (max_len == 1) {
    const long tot = (long)S * R;
    const int g1 = (int)((tot + 255) / 256 < 8192 ? (tot + 255) / 256 : 8192);
    MX_DISPATCH(dt_in, TI, MX_DISPATCH(dt_out, TO, mingru_step_kernel<TI, TO><<<g1, 256, 0, st>>>(
        (const TI*)zp, sz, (const TI*)xp, sx, (const TI*)gp, sg, z_bias, x_bias, state, cu, slot, pos, (TO*)out, S, R)));
    MX_RETURN_LAUNCH();
  }
  if (ab == nullptr || gy == nullptr) return (int)hipErrorInvalidValue;
  const long total = (long)T * R;
  const int gb = (int)((total + 255) / 256 < 8192 ? (total + 255) / 256 : 8192);
  MX_DISPATCH(dt_in, TI, mingru_gates_kernel<TI><<<gb, 256, 0, st>>>((const TI*)zp, sz, (const TI*)xp, sx, (const TI*)gp, sg,
                                                                     z_bias, x_bias, ab, gy, (long)T, R));
  dim3 grid((R + LRU_CH - 1) / LRU_CH, S);
  MX_DISPATCH(dt_out, TO, lru_scan_kernel<TO><<<grid, 256, 0, st>>>(ab, gy, R, (long)T, state, cu, slot, pos, (TO*)out, R));
  MX_RETURN_LAUNCH();
}
