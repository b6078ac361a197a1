// State-space (Mamba-2 form) mixer kernels over a flat batch of segments.
//
// A step's rows are `S` segments (a prompt chunk or one decoded token each): segment s owns rows
// cu[s] .. cu[s+1]-1, continues the sequence at position pos[cu[s]] and keeps its recurrent state
// in slot slot[s] (< 0: a padding row, skipped).  A segment that starts at position 0 starts from
// a zero state whatever its slot held before, so a slot needs no clearing when it is handed on.
//
//   conv:  u_t[c] = silu(b[c] + sum_k w[c][k] * in_{t-(K-1)+k}[c]),  inputs before the sequence are 0,
//          inputs before the chunk come from the slot's last K-1 inputs.
//   scan:  per head h (group g = h / (H / G)), state S [P][N] in f32:
//            dt = softplus(dt_raw + dt_bias[h]);  a = exp(-exp(A_log[h]) * dt)
//            S <- a * S + dt * x_t (outer) B_t;   y_t = S C_t + D[h] * x_t
//          u rows are laid out [x: H*P | B: G*N | C: G*N].
//          Steps with long segments, by the caller's choice, run those of SSD_LEAST tokens or more in chunks of 64 on the
//          f32 matrix instructions (ssd_scan_kernel); all else goes token by token (ssm_scan_kernel).
#include <type_traits>

#include "mx_common.h"

namespace {

constexpr int CONV_TT = 32;   // tokens per block of the convolution
constexpr int MAX_TAPS = 8;

// Both forms: the thread of a segment's first tile is the only one that reads the slot's history of its channels (a tile has more
// rows than the taps reach back), and it replaces it by the segment's last K-1 inputs, upward, reading entry j + n before it
// writes entry j.  (A launch of its own for that took 4.6 - 5.6 us behind each convolution.)

// grid (ceil(C/256), tiles of the segments, in y and z: one of them holds 65535 of 32 rows)
template <typename T>
__global__ void conv_silu_kernel(const T* __restrict__ in, long si, const float* __restrict__ w,
                                 const float* __restrict__ bias, const float* __restrict__ in_bias, int act, float* state,
                                 const int* __restrict__ cu, const int* __restrict__ slot, const int* __restrict__ pos,
                                 float* __restrict__ out, int S, int per, int C, int K) {
  int s, t0;
  if (!mx_tile_place<1>(cu, S, per, CONV_TT, blockIdx.z * gridDim.y + blockIdx.y, s, t0)) return;
  const int sl = slot[s];
  if (sl < 0) return;
  const int r0 = cu[s], n = cu[s + 1] - r0;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const bool fresh = pos[r0] == 0;
  float* st = state + (long)sl * (K - 1) * C;
  float wk[MAX_TAPS], win[MAX_TAPS];
  const float ib = in_bias != nullptr ? in_bias[c] : 0.f;   // added to every real input (the history holds biased inputs)
#pragma unroll
  for (int k = 0; k < MAX_TAPS; ++k) {
    wk[k] = k < K ? w[(long)c * K + k] : 0.f;
    win[k] = 0.f;
  }
  // win[k] holds the input at local index i - (K-1) + k for the current i
#pragma unroll
  for (int k = 0; k < MAX_TAPS - 1; ++k) {
    if (k < K - 1) {
      const int j = t0 - (K - 1) + k;          // local index, may be < 0
      win[k + 1] = j >= 0 ? ldf(in + (long)(r0 + j) * si + c) + ib : (fresh ? 0.f : st[(long)(K - 1 + j) * C + c]);
    }
  }
  if (t0 == 0)
    for (int j = 0; j < K - 1; ++j) {
      const int i = n - (K - 1) + j;             // local index of the input that lands in entry j
      st[(long)j * C + c] = i >= 0 ? ldf(in + (long)(r0 + i) * si + c) + ib : (fresh ? 0.f : st[(long)(j + n) * C + c]);
    }
  const float b = bias != nullptr ? bias[c] : 0.f;
  const int t1 = min(t0 + CONV_TT, n);
  for (int i = t0; i < t1; ++i) {
#pragma unroll
    for (int k = 0; k < MAX_TAPS - 1; ++k) win[k] = win[k + 1];
    // after the shift the newest input goes to tap K-1
    const float v = ldf(in + (long)(r0 + i) * si + c) + ib;
#pragma unroll
    for (int k = 0; k < MAX_TAPS; ++k) if (k == K - 1) win[k] = v;
    float acc = b;
#pragma unroll
    for (int k = 0; k < MAX_TAPS; ++k) if (k < K) acc += wk[k] * win[k];
    out[(long)(r0 + i) * C + c] = act == 1 ? mx_silu(acc) : acc;
  }
}

// The same for K = 4 taps and channels by fours, TT tokens of a segment per thread (grid ceil(C/1024)): every load of a thread, the
// next history's included, is issued before the first is used, so that a tile takes one trip to memory.
template <typename T, int TT>
__global__ void __launch_bounds__(256) conv4_kernel(const T* __restrict__ in, long si, const float* __restrict__ w,
                                                    const float* __restrict__ bias, const float* __restrict__ in_bias, int act,
                                                    float* state, const int* __restrict__ cu,
                                                    const int* __restrict__ slot, const int* __restrict__ pos,
                                                    float* __restrict__ out, int S, int per, int C) {
  static_assert(TT == 1 || TT >= 3, "a tile behind a segment's first reads three rows back; single-row tiles are for segments of one row");
  int s, t0;
  if (!mx_tile_place<1>(cu, S, per, TT, blockIdx.z * gridDim.y + blockIdx.y, s, t0)) return;
  const int sl = slot[s];
  if (sl < 0) return;
  const int r0 = cu[s], n = cu[s + 1] - r0;
  const int c = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (c >= C) return;
  const bool fresh = pos[r0] == 0, first = t0 == 0;
  float* st = state + (long)sl * 3 * C + c;
  const T* seg = in + (long)r0 * si + c;
  const mx_f32x4 zero = mx_f32x4{0.f, 0.f, 0.f, 0.f};
  mx_f32x4 x[TT + 3], h[3];              // x[k]: the input at local index t0 - 3 + k; h[j]: the next history
#pragma unroll
  for (int i = 0; i < TT; ++i) x[3 + i] = ldf4(seg + min(t0 + i, n - 1) * si);
#pragma unroll
  for (int k = 0; k < 3; ++k) x[k] = first ? (fresh ? zero : ldf4(st + (long)k * C)) : ldf4(seg + max(t0 - 3 + k, 0) * si);
  if (first)
#pragma unroll
    for (int j = 0; j < 3; ++j) h[j] = ldf4(seg + max(n - 3 + j, 0) * si);
  mx_f32x4 wk[4];                        // weights [C][4]: channel c + e, tap k
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const mx_f32x4 r = ldf4(w + 4L * (c + e));
#pragma unroll
    for (int k = 0; k < 4; ++k) wk[k][e] = r[k];
  }
  const mx_f32x4 ib = in_bias != nullptr ? ldf4(in_bias + c) : zero;   // added to every real input (not to the history)
  const mx_f32x4 b = bias != nullptr ? ldf4(bias + c) : zero;
  if (first) {                           // x[0 .. 2] is the history: entry j takes input n - 3 + j, or entry j + n of before
#pragma unroll
    for (int j = 0; j < 3; ++j) stf4(st + (long)j * C, n - 3 + j >= 0 ? h[j] + ib : (j + n == 1 ? x[1] : x[2]));
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] += ib;
  }
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    x[3 + i] += ib;
    mx_f32x4 y = b;
#pragma unroll
    for (int k = 0; k < 4; ++k) y += wk[k] * x[i + k];
    if (act == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = mx_silu(y[e]);
    }
    if (t0 + i < n) stf4(out + (long)(r0 + t0 + i) * C + c, y);
  }
}

// Sequential scan.  grid (ceil(P/PT), H, S), block PT * NS threads: thread (p, ns) keeps the NI
// consecutive state entries S[p][ns*NI .. ns*NI+NI-1] in registers (a wave's state loads and stores
// are contiguous runs of the slot's [P][N] record); the NS partial sums of y_t[p] are reduced
// inside the 16-lane row with DPP swaps.  N is padded to 16 * NI with zeros (B, C and the state
// entries past N stay 0), so the per-token loop has no bounds checks.  The rows of a chunk of TB
// tokens (B_t | C_t, the block's x_t, dt and the decay) are staged in LDS; the next chunk's rows
// are fetched into registers -- unconditional, clamped loads, issued back to back -- before the
// current chunk's TB dependent steps run, so the recurrence never waits on HBM.
constexpr int SCAN_NS = 16;       // lanes sharing one value channel
constexpr int SCAN_PT = 16;       // value channels per block (256 threads)
constexpr int SCAN_PF = 36;       // prefetch registers per thread: TB * 2N <= 256 * SCAN_PF
constexpr int SCAN_NT = SCAN_PT * SCAN_NS;

// sum over the 16 lanes of a DPP row, result in every lane: xor 1, xor 2 (quad permutes), then the
// mirrored 8-lane and 16-lane halves
__device__ __forceinline__ float row_sum16(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));   // row_half_mirror
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true));   // row_mirror
  return v;
}

// The sum over 64 entries of the state, four in each of 16 lanes, in the order of a lane of the scan below, which owns 4 NJ entries side by side:
// a run of NJ lanes passes its two partial sums on, then the runs meet as row_sum16 adds the scan's lanes.
template <int NJ>
__device__ __forceinline__ float run_sum(mx_f32x4 s, mx_f32x4 c, int ns) {
  float even = 0.f, odd = 0.f;
  const auto chain = [&] {
    even = fmaf(s[2], c[2], fmaf(s[0], c[0], even));
    odd = fmaf(s[3], c[3], fmaf(s[1], c[1], odd));
  };
  const auto from = [](float v, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), decltype(ctrl)::value, 0xF, 0xF, true));
  };
  chain();
#pragma unroll
  for (int hop = 1; hop < NJ; ++hop) {         // quad_perm [3,0,1,2]: the lane before
    even = from(even, std::integral_constant<int, 0x93>{});
    odd = from(odd, std::integral_constant<int, 0x93>{});
    if (ns % NJ == 0) even = odd = 0.f;
    chain();
  }
  float v = even + odd;
  if (NJ == 1) return row_sum16(v);
  if (NJ == 2) {                               // each pair's second lane has it: quad_perm [1,1,3,3], then pairs, eights, the row
    v = from(v, std::integral_constant<int, 0xF5>{});
    v += from(v, std::integral_constant<int, 0x4E>{});
  } else {
    v = from(v, std::integral_constant<int, 0xFF>{});
  }
  v += from(v, std::integral_constant<int, 0x141>{});
  return v + from(v, std::integral_constant<int, 0x140>{});
}

// A step of single rows (decode): a block takes a head, its threads 16 of the value channels at a time with 16 lanes by fours along
// the state's NJ 64s, up to 64 channels' states asked for at once; B and C, the same for all of them, stay in registers.  Bound by the
// state's bytes, which do not stay in the caches on either way: 64 rows of 64 heads of 64 x 128 46 us (5.8 TB/s; 48 where they stay, and
// the step's other launches longer: 8 layers 1157 / 1117, 17 rows 504 / 480), by the scan below, whose chunk of staged rows leaves room for three blocks a
// CU, 62; 17 rows of 32 heads 9.6, 13.4.  Every product, sum and rounding is that of the scan's single token, so that a row's results do not
// depend on which of the two its step takes: the lanes' passing on is free beside the bytes (44.2 us added up as the lanes lie, 44.4 so), and
// added up as they lie, values and states of 64 entries were 5 and 9 % further from 64 bits than the scan's.  (Entries side by side in a lane,
// as the scan reads them, break the loads past the caches into halves of lines: 69 us.)
template <typename TD, int NJ>
__global__ void __launch_bounds__(256)
ssm_step_kernel(const float* __restrict__ u, int C, const TD* __restrict__ dt_raw, long sdt, const float* __restrict__ dt_bias,
                const float* __restrict__ A_log, const float* __restrict__ Dp, float* __restrict__ state, const int* __restrict__ cu,
                const int* __restrict__ slot, const int* __restrict__ pos, float* __restrict__ y, int H, int P, int G) {
  constexpr int N = 64 * NJ, PU = NJ <= 2 ? 4 : 2;
  const int s = blockIdx.y, sl = slot[s];
  if (sl < 0) return;
  const long t = cu[s];
  if (cu[s + 1] - (int)t <= 0) return;
  const int h = blockIdx.x, ns = threadIdx.x & 15, pl = threadIdx.x >> 4, inner = H * P;
  const bool fresh = pos[t] == 0;
  const float* ur = u + t * C;
  float* sh = state + ((long)sl * H + h) * P * N + 4 * ns;
  const float* Br = ur + inner + (long)(h / (H / G)) * N + 4 * ns;
  mx_f32x4 B[NJ], Cv[NJ], S[PU][NJ];
  float x[PU];
  auto load = [&](int p0) {
#pragma unroll
    for (int i = 0; i < PU; ++i) {
      const int p = min(p0 + 16 * i + pl, P - 1);
      x[i] = ur[h * P + p];
#pragma unroll
      for (int j = 0; j < NJ; ++j) S[i][j] = fresh ? mx_f32x4{0.f, 0.f, 0.f, 0.f} : ldf4_once(sh + (long)p * N + 64 * j);
    }
  };
  load(0);
#pragma unroll
  for (int j = 0; j < NJ; ++j) B[j] = ldf4(Br + 64 * j), Cv[j] = ldf4(Br + (long)G * N + 64 * j);
  const float dt = mx_softplus(ldf(dt_raw + t * sdt + h) + dt_bias[h]), a = expf(-expf(A_log[h]) * dt), Dh = Dp[h];
  for (int p0 = 0; p0 < P; p0 += 16 * PU) {
    if (p0 > 0) load(p0);
#pragma unroll
    for (int i = 0; i < PU; ++i) {
      const int p = p0 + 16 * i + pl;
      const float dx = dt * x[i];
      float part[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i][j][e] = NJ == 1 ? fmaf(a, S[i][j][e], dx * B[j][e]) : fmaf(dx, B[j][e], a * S[i][j][e]);
        if (p < P) stf4_once(sh + (long)p * N + 64 * j, S[i][j]);
        part[j] = run_sum<NJ>(S[i][j], Cv[j], ns);
      }
      const float o = NJ == 4 ? (part[0] + part[1 % NJ]) + (part[2 % NJ] + part[3 % NJ]) : NJ == 2 ? part[0] + part[1 % NJ] : part[0];
      if (ns == 0 && p < P) y[t * inner + h * P + p] = fmaf(Dh, x[i], o);
    }
  }
}

// VEC: B | C rows are fetched and staged as 16-byte pieces (N, H*P and the row stride multiples of 4)
template <typename TD, int NI, bool VEC>
__global__ void __launch_bounds__(SCAN_NT) __attribute__((amdgpu_waves_per_eu(NI <= 8 ? 3 : 2)))   // blocks per CU that hide the step latency
ssm_scan_kernel(const float* __restrict__ u, int C, const TD* __restrict__ dt_raw, long sdt,
                const float* __restrict__ dt_bias, const float* __restrict__ A_log, const float* __restrict__ Dp,
                float* __restrict__ state, const int* __restrict__ cu, const int* __restrict__ slot,
                const int* __restrict__ pos, float* __restrict__ y, int H, int P, int N, int G, int TB, int below) {
  extern __shared__ __align__(16) float rows[];   // [TB][RW]: B[NP] | C[NP] | x[PT] | dt | decay | pad
  constexpr int NP = SCAN_NS * NI;                // padded state size
  constexpr int RW = 2 * NP + SCAN_PT + 4;
  const int s = blockIdx.z;
  const int sl = slot[s];
  if (sl < 0) return;
  const int h = blockIdx.y;
  const int tid = threadIdx.x;
  const int ns = tid % SCAN_NS;
  const int pl = tid / SCAN_NS;
  const int p0 = blockIdx.x * SCAN_PT;
  const int p = p0 + pl;
  const bool live = p < P;
  const int pc = live ? p : P - 1;
  const int r0 = cu[s], n = cu[s + 1] - r0;
  if (n <= 0 || n >= below) return;          // longer segments belong to ssd_scan_kernel
  const int g = h / (H / G);
  const bool fresh = pos[r0] == 0;
  const int inner = H * P;
  const int W2 = 2 * N;
  const int kb = ns * NI;                    // this lane's first state entry
  const bool vec = (NI % 4 == 0) && N == NP; // 16-byte state and LDS accesses
  float* sp = state + (((long)sl * H + h) * P + pc) * N;
  float S[NI];
  if (vec) {
#pragma unroll
    for (int i = 0; i < NI; i += 4) {
      const float4 v = fresh ? float4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const float4*>(sp + kb + i);
      S[i] = v.x;
      S[i + 1 < NI ? i + 1 : i] = v.y;
      S[i + 2 < NI ? i + 2 : i] = v.z;
      S[i + 3 < NI ? i + 3 : i] = v.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i) S[i] = (!fresh && kb + i < N) ? sp[kb + i] : 0.f;
  }
  const float A = -expf(A_log[h]);
  const float bias = dt_bias[h], Dh = Dp[h];
  // B_t | C_t of group g are 2N floats that are contiguous when G == 1, two runs otherwise
  const float* ub = u + inner + g * N;
  const long c_off = (long)(G - 1) * N;      // extra offset of the C run (col >= N)
  // per-thread walk over the chunk's TB x 2N elements (in pieces of UW floats) without divisions
  using U = std::conditional_t<VEC, float4, float>;
  constexpr int UW = VEC ? 4 : 1, PFN = SCAN_PF / UW;
  const int W2u = W2 / UW;
  const int step_t = SCAN_NT / W2u, step_c = SCAN_NT % W2u;
  const int tt0 = tid / W2u, col0 = tid % W2u;
  U pf[PFN];
  float pfx[2], pfd = 0.f;

  // (32-bit element offsets from the block-uniform bases: the launcher checks rows * C < 2^31)
  auto fetch = [&](int c0) {                 // rows c0 .. c0+TB-1 of the segment -> registers
    const int last = n - 1 - c0;             // rows past the segment re-read its last row (never used)
    int tt = tt0, col = col0;
#pragma unroll
    for (int j = 0; j < PFN; ++j) {
      const int r = r0 + c0 + min(tt, last);
      const int ce = col * UW;
      pf[j] = *reinterpret_cast<const U*>(ub + (unsigned)(r * C + ce + (ce >= N ? (int)c_off : 0)));
      col += step_c;
      tt += step_t;
      if (col >= W2u) {
        col -= W2u;
        ++tt;
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = tid + j * SCAN_NT;       // (token, channel) of the block's x
      const int tx = e / SCAN_PT, px = p0 + e % SCAN_PT;
      pfx[j] = u[(unsigned)((r0 + c0 + min(tx, last)) * C + h * P + min(px, P - 1))];
    }
    pfd = ldf(dt_raw + (r0 + c0 + min(tid, last)) * sdt + h);
  };

  if (n == 1) {
    // a decoded token: no staging -- every lane reads its own B / C entries and the row's scalars
    const float* ur = u + (long)r0 * C;
    const float dt = mx_softplus(ldf(dt_raw + (long)r0 * sdt + h) + bias);
    const float a = expf(A * dt);
    const float x = ur[h * P + pc];
    const float dx = dt * x;
    const float* Br = ub + (long)r0 * C + kb;
    const float* Cr = Br + N + c_off;
    float acc0 = 0.f, acc1 = 0.f;
    if (vec && (inner & 3) == 0 && (C & 3) == 0) {      // the row's B / C runs are 16-byte aligned too
#pragma unroll
      for (int i = 0; i < NI; i += 4) {
        const float4 b4 = *reinterpret_cast<const float4*>(Br + i), c4 = *reinterpret_cast<const float4*>(Cr + i);
        const float bb[4] = {b4.x, b4.y, b4.z, b4.w}, cc[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = i + j < NI ? i + j : i;
          S[k] = a * S[k] + dx * bb[j];
          if (j & 1) acc1 += S[k] * cc[j]; else acc0 += S[k] * cc[j];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (kb + i < N) {
          S[i] = a * S[i] + dx * Br[i];
          acc0 += S[i] * Cr[i];
        }
    }
    const float acc = row_sum16(acc0 + acc1);
    if (live) {
      if (ns == 0) y[(long)r0 * inner + h * P + p] = acc + Dh * x;
      if (vec) {
#pragma unroll
        for (int i = 0; i < NI; i += 4)
          *reinterpret_cast<float4*>(sp + kb + i) =
              float4{S[i], S[i + 1 < NI ? i + 1 : i], S[i + 2 < NI ? i + 2 : i], S[i + 3 < NI ? i + 3 : i]};
      } else {
#pragma unroll
        for (int i = 0; i < NI; ++i)
          if (kb + i < N) sp[kb + i] = S[i];
      }
    }
    return;
  }
  if (N != NP)                               // the padding columns of B and C stay zero
    for (int e = tid; e < TB * RW; e += SCAN_NT) rows[e] = 0.f;
  fetch(0);
  for (int c0 = 0; c0 < n; c0 += TB) {
    const int m = min(TB, n - c0);
    __syncthreads();                         // the previous chunk's readers are done
    {
      int tt = tt0, col = col0;
#pragma unroll
      for (int j = 0; j < PFN; ++j) {
        const int ce = col * UW;
        if (tt < TB) *reinterpret_cast<U*>(rows + tt * RW + (ce >= N ? ce - N + NP : ce)) = pf[j];
        col += step_c;
        tt += step_t;
        if (col >= W2u) {
          col -= W2u;
          ++tt;
        }
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int e = tid + j * SCAN_NT;
        if (e / SCAN_PT < TB) rows[(e / SCAN_PT) * RW + 2 * NP + e % SCAN_PT] = pfx[j];
      }
      if (tid < TB) {
        const float dt = mx_softplus(pfd + bias);
        rows[tid * RW + 2 * NP + SCAN_PT] = dt;
        rows[tid * RW + 2 * NP + SCAN_PT + 1] = expf(A * dt);
      }
    }
    __syncthreads();
    if (c0 + TB < n) fetch(c0 + TB);
    for (int t = 0; t < m; ++t) {
      const float* row = rows + t * RW;
      const float x = row[2 * NP + pl];
      const float2 da = *reinterpret_cast<const float2*>(row + 2 * NP + SCAN_PT);
      const float dx = da.x * x;
      float Bv[NI], Cv[NI];
      if (NI % 4 == 0) {
#pragma unroll
        for (int i = 0; i < NI; i += 4) {
          const float4 b4 = *reinterpret_cast<const float4*>(row + kb + i);
          const float4 c4 = *reinterpret_cast<const float4*>(row + NP + kb + i);
          Bv[i] = b4.x; Bv[i + 1 < NI ? i + 1 : i] = b4.y; Bv[i + 2 < NI ? i + 2 : i] = b4.z; Bv[i + 3 < NI ? i + 3 : i] = b4.w;
          Cv[i] = c4.x; Cv[i + 1 < NI ? i + 1 : i] = c4.y; Cv[i + 2 < NI ? i + 2 : i] = c4.z; Cv[i + 3 < NI ? i + 3 : i] = c4.w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          Bv[i] = row[kb + i];
          Cv[i] = row[NP + kb + i];
        }
      }
      float acc = 0.f, acc1 = 0.f;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        S[i] = da.y * S[i] + dx * Bv[i];
        if (i & 1) acc1 += S[i] * Cv[i]; else acc += S[i] * Cv[i];
      }
      acc = row_sum16(acc + acc1);
      if (ns == 0 && live) y[(long)(r0 + c0 + t) * inner + h * P + p] = acc + Dh * x;
    }
  }
  if (live) {
    if (vec) {
#pragma unroll
      for (int i = 0; i < NI; i += 4)
        *reinterpret_cast<float4*>(sp + kb + i) =
            float4{S[i], S[i + 1 < NI ? i + 1 : i], S[i + 2 < NI ? i + 2 : i], S[i + 3 < NI ? i + 3 : i]};
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (kb + i < N) sp[kb + i] = S[i];
    }
  }
}

// ---- chunked form ------------------------------------------------------------------------------------------------
// With c_t the running sum of log decays A dt inside a chunk of 64 tokens and S the state before it,
//     y_t = e^(c_t) C_t S^T + sum_(s<=t) (C_t . B_s) e^(c_t - c_s) dt_s x_s + D x_t
//     S  <- e^(c_63) S + sum_s e^(c_63 - c_s) dt_s x_s B_s^T
// all in f32 (v_mfma_f32_16x16x4_f32; the sums c in f64, so that their differences are good to f32 however far the
// chunk decays).  Three launches leave to the serial one only products: ssd_scores_kernel makes C . B of a group, which its
// heads share, and B and C in operand order; ssd_decay_kernel the factors of every chunk and head, M[t][s] = (C_t . B_s)
// e^(c_t - c_s) dt_s for s <= t (else 0), E[t] = e^(c_t), F[s] = e^(c_63 - c_s) dt_s; then a block of ssd_scan_kernel owns 16
// value channels of one head and walks the chunks of its segment: wave w owns tokens 16 w .. 16 w + 15 of the outputs and
// N / 4 columns of the state, which the waves exchange through LDS, one barrier per chunk.  Every operand but the values is read
// from memory in the register layout of its product -- K index 16 j + 4 g + e of step (j, e) for lane group g on both sides --
// and the loads of the next chunk are issued as soon as the registers are free; the values come one 16-byte load a thread, two
// chunks ahead, and turn through LDS.  Bound by the chunk's chain (1.1 us of its 2.6 to 4 are products: 80 per wave);
// 2 prompts of 2048, 64 heads of 64 x 128, 2 groups: 158 us in all; with C and the values read from their rows, 64 bytes
// each and far apart, 183; one prompt 106 and 121.  (Waves of their own for the state and the outputs: 3 % less for one prompt,
// 20 % more for three uneven ones.)
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int SSD_L = 64;           // tokens per chunk
constexpr int SSD_LEAST = 32;       // shorter segments of a step in chunks go token by token: a chunk costs about 20 steps

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Scratch of a chunk: per group C . B [64][64] (s up to t's tile of 16), B in operand order [N / 16][4][64 lanes][4 tokens] and C
// in operand order [4][N / 16][64 lanes][4 columns]; per head M in operand order [10 tiles (w, j <= w)][64 lanes][4], E, F.
constexpr int SSD_HEAD = 10 * 256 + 2 * SSD_L;
__host__ __device__ inline long ssd_group_floats(int N) { return 64L * SSD_L + 2 * 64L * N; }
__host__ __device__ inline long ssd_chunk_floats(int N, int G, int H) { return G * ssd_group_floats(N) + (long)H * SSD_HEAD; }

// max_len is a bound: the only segment of a step may be of any length, and needs no fourth launch whatever it is
__host__ __device__ inline int ssd_least(int S) { return S == 1 ? 1 : SSD_LEAST; }

// The chunk that segment s, from row r0 on, starts at: no two segments of SSD_LEAST rows or more share one, and the shorter
// ones, which have none, do not move it by more than the rows before it allow.
__host__ __device__ inline int ssd_first(int r0, int s) { return r0 / SSD_L + (s < r0 / SSD_LEAST ? s : r0 / SSD_LEAST); }

// all chunks of S segments in T rows
__host__ __device__ inline int ssd_chunks(int T, int S) { return ssd_first(T, S) > 1 ? ssd_first(T, S) : 1; }

// the last segment that starts at or before chunk ci
__device__ __forceinline__ int ssd_segment(const int* cu, int S, int ci) {
  int s = 0;
  for (int lo = 0, hi = S; lo < hi;) {
    const int mid = (lo + hi) >> 1;
    if (ssd_first(cu[mid], mid) <= ci) {
      s = mid;
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  return s;
}

// grid (ssd_chunks(T, S), G)
template <int NTW>
__global__ void __launch_bounds__(256, 2) ssd_scores_kernel(const float* __restrict__ u, int C, const int* __restrict__ cu,
                                                            const int* __restrict__ slot, float* __restrict__ ws, int S, int H,
                                                            int inner, int G) {
  constexpr int N = 64 * NTW, NJ = N / 16;
  const int ci = blockIdx.x, grp = blockIdx.y, s = ssd_segment(cu, S, ci);
  const int r0 = cu[s], n = cu[s + 1] - r0, c0 = (ci - ssd_first(r0, s)) * SSD_L;
  if (slot[s] < 0 || n < ssd_least(S) || c0 < 0 || c0 >= n) return;
  float* cb = ws + ci * ssd_chunk_floats(N, G, H) + grp * ssd_group_floats(N);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const float* ub = u + inner + grp * N + 4 * g;
  const float* cr = ub + (long)G * N + (long)(r0 + min(c0 + 16 * w + c, n - 1)) * C;
  f32x4 cv[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) cv[j] = *reinterpret_cast<const f32x4*>(cr + 16 * j);
  for (int st = 0; st <= w; ++st) {
    const float* br = ub + (long)(r0 + min(c0 + 16 * st + c, n - 1)) * C;
    f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(br + 16 * j);
      a0 = mma4(cv[j][0], bv[0], a0);
      a1 = mma4(cv[j][1], bv[1], a1);
      a0 = mma4(cv[j][2], bv[2], a0);
      a1 = mma4(cv[j][3], bv[3], a1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) cb[(16 * w + 4 * g + r) * SSD_L + 16 * st + c] = a0[r] + a1[r];
  }
  float* ct = cb + SSD_L * SSD_L + 64 * N;
#pragma unroll
  for (int j = 0; j < NJ; ++j) *reinterpret_cast<f32x4*>(ct + ((w * NJ + j) * 64 + lane) * 4) = cv[j];
  // B: wave w's tokens 16 w + 4 g + e, column 16 i + c
  float* bt = cb + SSD_L * SSD_L;
  const float* bp = u + inner + grp * N + c;
#pragma unroll
  for (int i = 0; i < NJ; ++i) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = bp[(long)(r0 + min(c0 + 16 * w + 4 * g + e, n - 1)) * C + 16 * i];
    *reinterpret_cast<f32x4*>(bt + ((i * 4 + w) * 64 + lane) * 4) = v;
  }
}

// grid (ssd_chunks(T, S), H)
template <typename TD>
__global__ void __launch_bounds__(256) ssd_decay_kernel(const TD* __restrict__ dt_raw, long sdt,
                                                        const float* __restrict__ dt_bias, const float* __restrict__ A_log,
                                                        const int* __restrict__ cu, const int* __restrict__ slot,
                                                        float* __restrict__ ws, int S, int H, int G, int N) {
  __shared__ double cums[4][SSD_L];      // a copy per wave
  __shared__ float dts[4][SSD_L];
  const int ci = blockIdx.x, h = blockIdx.y, s = ssd_segment(cu, S, ci);
  const int r0 = cu[s], n = cu[s + 1] - r0, c0 = (ci - ssd_first(r0, s)) * SSD_L;
  if (slot[s] < 0 || n < ssd_least(S) || c0 < 0 || c0 >= n) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const float A = -expf(A_log[h]);
  const float raw = ldf(dt_raw + (long)(r0 + min(c0 + lane, n - 1)) * sdt + h);
  const float dt = c0 + lane < n ? mx_softplus(raw + dt_bias[h]) : 0.f;
  double a = (double)(A * dt);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double v = __shfl_up(a, o, 64);
    if (lane >= o) a += v;
  }
  cums[w][lane] = a;
  dts[w][lane] = dt;
  __builtin_amdgcn_wave_barrier();
  const double* cw = cums[w];
  float* chunk = ws + ci * ssd_chunk_floats(N, G, H);
  const float* cb = chunk + h / (H / G) * ssd_group_floats(N) + (16 * w + c) * SSD_L + 4 * g;
  float* out = chunk + G * ssd_group_floats(N) + (long)h * SSD_HEAD;
  const double ct = cw[16 * w + c];
  for (int j = 0; j <= w; ++j) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(cb + 16 * j);
    f32x4 m;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * j + 4 * g + e;
      m[e] = t <= 16 * w + c ? v[e] * expf((float)(ct - cw[t])) * dts[w][t] : 0.f;
    }
    *reinterpret_cast<f32x4*>(out + ((w * (w + 1) / 2 + j) * 64 + lane) * 4) = m;
  }
  if (w == 0) {
    out[2560 + lane] = expf((float)a);
    out[2560 + SSD_L + lane] = dt * expf((float)(cw[SSD_L - 1] - a));
  }
}

// grid (H, P / 16, S): the value blocks of a head on one chiplet, whose cache then holds the chunk's factors
template <int NTW>
__global__ void __launch_bounds__(256, NTW == 4 ? 1 : 2)
ssd_scan_kernel(const float* __restrict__ u, int C, const float* __restrict__ Dp, float* __restrict__ state,
                const float* __restrict__ ws, const int* __restrict__ cu, const int* __restrict__ slot,
                const int* __restrict__ pos, float* __restrict__ y, int H, int P, int G) {
  constexpr int N = 64 * NTW, NJ = N / 16;
  __shared__ __attribute__((aligned(16))) float sbuf[2][16][N + 4];   // the state, [p][n]: rows 4 banks apart
  __shared__ __attribute__((aligned(16))) float xbuf[2][16][SSD_L + 4];   // a chunk's values, [p][token]
  const int s = blockIdx.z, h = blockIdx.x, p0 = blockIdx.y * 16;
  const int sl = slot[s], r0 = cu[s], n = cu[s + 1] - r0;
  if (sl < 0 || n < ssd_least(gridDim.z)) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const int grp = h / (H / G), inner = H * P, last = (n - 1) / SSD_L;
  const float Dh = Dp[h];
  const long step = ssd_chunk_floats(N, G, H);
  const float* base = ws + (long)ssd_first(r0, s) * step;
  const float* bbase = base + grp * ssd_group_floats(N) + SSD_L * SSD_L + (NTW * w * 256 + lane) * 4;
  const float* hbase = base + G * ssd_group_floats(N) + (long)h * SSD_HEAD;
  const int tok = threadIdx.x >> 2, xp = threadIdx.x & 3;              // the token and the four channels whose values this thread fetches
  const float* ux = u + (long)r0 * C + h * P + p0 + 4 * xp;
  const float* cbase = base + grp * ssd_group_floats(N) + SSD_L * SSD_L + 64 * N + (NJ * w * 64 + lane) * 4;
  float* sp = state + (((long)sl * H + h) * P + p0 + 4 * g) * N + 16 * NTW * w + c;
  float* yp = y + (long)(r0 + 16 * w + 4 * g) * inner + h * P + p0 + c;

  f32x4 st[NTW];                          // S[p0 + 4 g + r][16 (NTW w + i) + c]
#pragma unroll
  for (int i = 0; i < NTW; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      st[i][r] = pos[r0] == 0 ? 0.f : sp[(long)r * N + 16 * i];
      sbuf[0][4 * g + r][16 * (NTW * w + i) + c] = st[i][r];
    }

  f32x4 cv[NJ], mv[4], xv[4], bv[NTW][4], fv[4], ev;
  float keep;
  auto load_c = [&](int k) {              // k: the chunk (behind the end: the last one again)
    const float* p = cbase + min(k, last) * step;
#pragma unroll
    for (int j = 0; j < NJ; ++j) cv[j] = *reinterpret_cast<const f32x4*>(p + 256 * j);
  };
  auto load_m = [&](int k) {
    const float* p = hbase + min(k, last) * step;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= w) mv[j] = *reinterpret_cast<const f32x4*>(p + ((w * (w + 1) / 2 + j) * 64 + lane) * 4);
    ev = *reinterpret_cast<const f32x4*>(p + 2560 + 16 * w + 4 * g);
  };
  auto load_b = [&](int k) {
    const float* p = bbase + min(k, last) * step;
    const float* f = hbase + min(k, last) * step + 2560;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      fv[j] = *reinterpret_cast<const f32x4*>(f + SSD_L + 16 * j + 4 * g);
#pragma unroll
      for (int i = 0; i < NTW; ++i) bv[i][j] = *reinterpret_cast<const f32x4*>(p + (i * 4 + j) * 256);
    }
    keep = f[SSD_L - 1];
  };
  f32x4 xr;
  auto load_x = [&](int k) { xr = *reinterpret_cast<const f32x4*>(ux + (long)min(k * SSD_L + tok, n - 1) * C); };
  auto put_x = [&](int k) {
#pragma unroll
    for (int e = 0; e < 4; ++e) xbuf[k & 1][4 * xp + e][tok] = xr[e];
  };
  load_x(0);
  load_c(0);
  load_m(0);
  load_b(0);
  put_x(0);
  load_x(1);
  for (int k = 0; k <= last; ++k) {
    const int b = k & 1, left = n - k * SSD_L;
    __syncthreads();                      // the state of the last chunk is in sbuf[b], this one's values in xbuf[b]
#pragma unroll
    for (int j = 0; j < 4; ++j) xv[j] = *reinterpret_cast<const f32x4*>(&xbuf[b][c][16 * j + 4 * g]);
    put_x(k + 1);
    load_x(k + 2);
    // a value that is not finite spoils the tokens from its own on and its row of the state, nothing before
    int bad = SSD_L;
    const f32x4 xt = w == 0 ? xv[0] : (w == 1 ? xv[1] : (w == 2 ? xv[2] : xv[3]));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (left < SSD_L) {
#pragma unroll
        for (int e = 0; e < 4; ++e) xv[j][e] = 16 * j + 4 * g + e < left ? xv[j][e] : 0.f;
      }
      const int at = mx_drop_nonfinite(xv[j], g);
      bad = min(bad, at < 16 ? 16 * j + at : SSD_L);
    }
    // what the state before the chunk gives
    f32x4 y0 = {0.f, 0.f, 0.f, 0.f}, y1 = y0;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const f32x4 sv = *reinterpret_cast<const f32x4*>(&sbuf[b][c][16 * j + 4 * g]);
      y0 = mma4(cv[j][0], sv[0], y0);
      y1 = mma4(cv[j][1], sv[1], y1);
      y0 = mma4(cv[j][2], sv[2], y0);
      y1 = mma4(cv[j][3], sv[3], y1);
    }
    load_c(k + 1);
    y0 = (y0 + y1) * ev;
    // the chunk's own tokens up to this one
    y1 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j > w) continue;
      y0 = mma4(mv[j][0], xv[j][0], y0);
      y1 = mma4(mv[j][1], xv[j][1], y1);
      y0 = mma4(mv[j][2], xv[j][2], y0);
      y1 = mma4(mv[j][3], xv[j][3], y1);
    }
    load_m(k + 1);
    y0 += y1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * w + 4 * g + r;
      y0[r] = t >= bad ? NAN : y0[r] + Dh * xt[r];
      if (t < left) yp[(long)r * inner] = y0[r];
    }
    yp += (long)SSD_L * inner;
    // the state after the chunk
#pragma unroll
    for (int i = 0; i < NTW; ++i) st[i] *= keep;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 a = xv[j] * fv[j];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < NTW; ++i) st[i] = mma4(a[e], bv[i][j][e], st[i]);
    }
    load_b(k + 1);
    if (__any(bad < SSD_L)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool spoilt = __shfl(bad, 4 * g + r, 64) < SSD_L;
#pragma unroll
        for (int i = 0; i < NTW; ++i) st[i][r] = spoilt ? NAN : st[i][r];
      }
    }
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) sbuf[b ^ 1][4 * g + r][16 * (NTW * w + i) + c] = st[i][r];
  }
#pragma unroll
  for (int i = 0; i < NTW; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) sp[(long)r * N + 16 * i] = st[i][r];
}

}  // namespace

// in: [rows, C] slice (row stride si) of the in-projection; out: f32 [rows, C]; state f32 [slots, K-1, C]
// act: 0 none, 1 SiLU; in_bias (optional, [C]) is added to every input before the convolution; rows: those of the step
// Four taps go by four channels (conv4_kernel), tokens per thread by size: the fewer the shorter a tile's way, the more the fewer
// halo rows are read again once memory is the bound, and single rows need no tile (bf16, us, one channel and 32 tokens a thread in
// turn / 1 or 4 tokens / 8 / 16: 64 single rows of 4608 4.8 / 4.1, 512 20.4 / 12.4; one segment of 100 rows 11.8 / 4.4 / 5.6 / 8.1, 400
// 12.7 / 5.9 / 6.5 / 8.9, 800 14.2 / 9.3 / 9.4 / 10.2, 2048 22.9 / 19.3 / 18.2 / 19.6; 5065 rows behind their projection 41.4 with four
// channels and 32 tokens in turn, here by 8 38.9).
MX_API int mx_conv_act(const void* in, long si, int dt, const float* w, const float* bias, const float* in_bias, int act,
                       float* state, const int* cu, const int* slot, const int* pos, float* out, int S, int max_len,
                       int rows, int C, int K, hipStream_t st) {
  if (S <= 0 || max_len <= 0) return 0;
  if (K < 1 || K > MAX_TAPS || act < 0 || act > 1) return (int)hipErrorInvalidValue;
  auto grid = [&](int nx, int tt) {
    const int tiles = mx_tile_count(S, rows, max_len, tt, 4), tz = (tiles + 65534) / 65535;
    return dim3(nx, (tiles + tz - 1) / tz, tz);
  };
  if (K == 4 && C % 4 == 0 && mx_by_four(in, si, dt) &&
      ((size_t)w | (size_t)bias | (size_t)in_bias | (size_t)state | (size_t)out) % 16 == 0) {
#define CONV4(TT)                                                                                                                  \
  MX_DISPATCH(dt, TY, conv4_kernel<TY, TT><<<grid((C / 4 + 255) / 256, TT), 256, 0, st>>>((const TY*)in, si, w, bias, in_bias, act, state, cu, \
                                                                                          slot, pos, out, S, mx_tile_per(S, rows, max_len, TT, 4), C))
    const long size = (long)rows * C;
    if (max_len == 1) CONV4(1);
    else if (size < 8000000 || rows < 8L * S) CONV4(4);
    else CONV4(8);
#undef CONV4
  } else {
    MX_DISPATCH(dt, TT, conv_silu_kernel<TT><<<grid((C + 255) / 256, CONV_TT), 256, 0, st>>>((const TT*)in, si, w, bias, in_bias, act, state, cu,
                                                                   slot, pos, out, S, mx_tile_per(S, rows, max_len, CONV_TT, 4), C, K));
  }
  MX_RETURN_LAUNCH();
}

MX_API int mx_conv_silu(const void* in, long si, int dt, const float* w, const float* bias, float* state,
                        const int* cu, const int* slot, const int* pos, float* out, int S, int max_len, int rows, int C, int K,
                        hipStream_t st) {
  return mx_conv_act(in, si, dt, w, bias, nullptr, 1, state, cu, slot, pos, out, S, max_len, rows, C, K, st);
}

// u f32 [rows, C = H*P + 2*G*N]; dt_raw [rows, H] slice (stride sdt, type dt_code); state f32
// [slots, H, P, N]; y f32 [rows, H*P]; max_len: no segment is longer; ws: f32 scratch of
// max(1, rows / 64 + min(S, rows / 32)) * ssd_chunk_floats(N, G, H) values for the chunked form, or null (token by token).
// The chunked form takes states of 64, 128 or 256 columns, value sizes in whole tiles of 16 and 16-byte rows.
MX_API int mx_ssm_scan(const float* u, int C, const void* dt_raw, long sdt, int dt_code, const float* dt_bias,
                       const float* A_log, const float* D, float* state, const int* cu, const int* slot,
                       const int* pos, float* y, int S, int max_len, int H, int P, int N, int G, int cu_rows_bound,
                       float* ws, hipStream_t st) {
  if (S <= 0) return 0;
  if (N > SCAN_NS * 16 || G < 1 || H % G) return (int)hipErrorInvalidValue;
  if ((long)cu_rows_bound * C >= (1L << 31)) return (int)hipErrorInvalidValue;
  const bool vecu = (N % 4 == 0) && ((H * P) % 4 == 0) && (C % 4 == 0);
  const bool chunked = ws != nullptr && max_len >= SSD_LEAST && (N == 64 || N == 128 || N == 256) && P % 16 == 0 && vecu &&
                       ((size_t)u | (size_t)ws) % 16 == 0 && H <= 65535 && S <= 65535;
  if (chunked) {
    const int chunks = ssd_chunks(cu_rows_bound, S);
#define SSD(NTW)                                                                                                 \
  do {                                                                                                           \
    ssd_scores_kernel<NTW><<<dim3(chunks, G), 256, 0, st>>>(u, C, cu, slot, ws, S, H, H * P, G);                 \
    MX_DISPATCH(dt_code, TT, ssd_decay_kernel<TT><<<dim3(chunks, H), 256, 0, st>>>(                              \
        (const TT*)dt_raw, sdt, dt_bias, A_log, cu, slot, ws, S, H, G, N));                                      \
    ssd_scan_kernel<NTW><<<dim3(H, P / 16, S), 256, 0, st>>>(u, C, D, state, ws, cu, slot, pos, y, H, P, G);     \
  } while (0)
    if (N == 64) SSD(1);
    else if (N == 128) SSD(2);
    else SSD(4);
#undef SSD
    const int rc = (int)hipGetLastError();
    if (rc || S == 1) return rc;
  }
  if (max_len == 1 && (N == 64 || N == 128 || N == 256) && vecu && ((size_t)u | (size_t)state) % 16 == 0 && S <= 65535) {
#define SSM_STEP(NJ)                                                                                                               \
  MX_DISPATCH(dt_code, TT, ssm_step_kernel<TT, NJ><<<dim3(H, S), 256, 0, st>>>(u, C, (const TT*)dt_raw, sdt, dt_bias, A_log, D, state, cu, \
                                                                               slot, pos, y, H, P, G))
    if (N == 64) SSM_STEP(1);
    else if (N == 128) SSM_STEP(2);
    else SSM_STEP(4);
#undef SSM_STEP
    MX_RETURN_LAUNCH();
  }
  const int below = chunked ? SSD_LEAST : 0x7fffffff;
  dim3 grid((P + SCAN_PT - 1) / SCAN_PT, H, S);
  int TB = (SCAN_NT * SCAN_PF) / (2 * N);
  TB = TB > 32 ? 32 : TB;
  if (TB < 1) return (int)hipErrorInvalidValue;
  const int need = (N + SCAN_NS - 1) / SCAN_NS;         // state entries per lane, rounded up to 1, 2, 4, 8, 16
#define MX_SCAN(NI)                                                                                          \
  do {                                                                                                       \
    const size_t lds = (size_t)TB * (2 * SCAN_NS * NI + SCAN_PT + 4) * sizeof(float);                        \
    if (vecu)                                                                                                \
      MX_DISPATCH(dt_code, TT, ssm_scan_kernel<TT, NI, true><<<grid, SCAN_NT, lds, st>>>(                    \
          u, C, (const TT*)dt_raw, sdt, dt_bias, A_log, D, state, cu, slot, pos, y, H, P, N, G, TB, below)); \
    else                                                                                                     \
      MX_DISPATCH(dt_code, TT, ssm_scan_kernel<TT, NI, false><<<grid, SCAN_NT, lds, st>>>(                   \
          u, C, (const TT*)dt_raw, sdt, dt_bias, A_log, D, state, cu, slot, pos, y, H, P, N, G, TB, below)); \
  } while (0)
  if (need <= 1) MX_SCAN(1);
  else if (need <= 2) MX_SCAN(2);
  else if (need <= 4) MX_SCAN(4);
  else if (need <= 8) MX_SCAN(8);
  else MX_SCAN(16);
#undef MX_SCAN
  MX_RETURN_LAUNCH();
}
