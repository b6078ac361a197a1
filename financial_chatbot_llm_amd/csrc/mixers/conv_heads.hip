// Short causal convolution of projected query, key and value heads, with what follows it up to attention:
//
//   y_t[c] = sum_j w[c][j] * u_(t - (K-1) + j)[c]      per channel, zeros before the sequence's start, no activation
//   q, k:  y / sqrt(mean(y^2) + eps) * weight[D]       per head, the weight shared by the heads (null: no norm)
//   q:     times 1 + coef * ln(floor((p + 1) / every) + 1) at position p (coef 0: none)  -> qout [T, H*D]
//   k, v:  -> cache row slots[t] of [k: G*D | v: G*P]
//
// over a flat batch of segments (prompt chunks and single decoded tokens alike).  Segment s keeps its last K-1
// projected inputs in slot slot[s] of `state` (f32 [slots, K-1, C]); a segment that starts at position 0 starts from
// zeros whatever the slot held.  G = 0: queries only (a layer that reads another layer's keys and values).
//
// A wave owns one head and TT consecutive rows of a segment: all TT + K - 1 input rows and the slot's next history are fetched
// before the first is used (the loads overlap), the convolution runs from registers and the norms of four rows are reduced side by side.
// Only the wave of a segment's first tile reads the slot's history (TT >= K - 1), and it is the one that replaces it.
#include "mx_common.h"

namespace {

constexpr int CH_WAVES = 4;

// VE adjacent channels per lane and access, NC accesses per row, up to KM taps
template <typename T, int VE, int NC, int KM, int TT>
__global__ void __launch_bounds__(CH_WAVES * 64)
conv_heads_kernel(const T* __restrict__ in, long si, const float* __restrict__ w, int K, float* state,
                  const float* __restrict__ qw, const float* __restrict__ kw, float eps, float tcoef, int tevery,
                  const int* __restrict__ cu, const int* __restrict__ slot, const int* __restrict__ pos,
                  const int* __restrict__ slots, T* __restrict__ cache, T* __restrict__ qout, int S, int per, int H, int G, int D, int P) {
  static_assert(TT == 1 || TT >= KM - 1, "tiles behind the first must not reach the slot's history; single-row tiles are for segments of one row");
  constexpr int RB = TT < 4 ? TT : 4;
  typedef T vt __attribute__((ext_vector_type(VE)));
  constexpr int NV = NC * VE;
  int s, t0;
  const int unit = blockIdx.y * CH_WAVES + (threadIdx.x >> 6);
  if (unit >= H + 2 * G || !mx_tile_place<1>(cu, S, per, TT, blockIdx.x, s, t0)) return;     // wave-uniform, no block barrier below
  const int r0 = cu[s], n = cu[s + 1] - r0;
  const int lane = threadIdx.x & 63;
  const bool isq = unit < H, isv = unit >= H + G;
  const int nd = isv ? P : D;
  const int col = isq ? unit * D : (isv ? (H + G) * D + (unit - H - G) * P : unit * D);   // channels are q | k | v
  const int C = (H + G) * D + G * P;
  const int sl = slot[s];
  const bool fresh = sl < 0 || pos[r0] == 0;
  float* st = state + (sl < 0 ? 0 : (long)sl * (K - 1) * C) + col;
  const int pad = KM - K;                                // taps are aligned to the end of the KM-wide window

  float x[TT + KM - 1][NV], wk[KM][NV], h[KM <= 8 ? KM - 1 : 1][NV];
  const bool first = t0 == 0, keep = first && sl >= 0;
  // every load is issued before the first is used: rows behind the segment's end read its last one, and are not used
#pragma unroll
  for (int r = 0; r < TT + KM - 1; ++r) {
    const int j = t0 - (KM - 1) + r;                     // row of the segment, < 0: history
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = (c * 64 + lane) * VE;
#pragma unroll
      for (int e = 0; e < VE; ++e) x[r][c * VE + e] = 0.f;
      if (d < nd) {
        if (r >= KM - 1 || !first) {
          const vt v = *reinterpret_cast<const vt*>(in + (long)(r0 + max(min(j, n - 1), 0)) * si + col + d);
#pragma unroll
          for (int e = 0; e < VE; ++e) x[r][c * VE + e] = (float)v[e];
        } else if (!fresh && K - 1 + j >= 0) {
#pragma unroll
          for (int e = 0; e < VE; ++e) x[r][c * VE + e] = st[(long)(K - 1 + j) * C + d + e];
        }
      }
    }
  }
  if (KM <= 8 && keep)
#pragma unroll
    for (int e = 0; e < (KM <= 8 ? KM - 1 : 0); ++e)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int d = (c * 64 + lane) * VE, i = n - (K - 1) + e;
#pragma unroll
        for (int q = 0; q < VE; ++q) h[e][c * VE + q] = 0.f;
        if (d < nd && e < K - 1) {
#pragma unroll
          for (int q = 0; q < VE; ++q)
            h[e][c * VE + q] = i >= 0 ? ldf(in + (long)(r0 + i) * si + col + d + q) : (fresh ? 0.f : st[(long)(e + n) * C + d + q]);
        }
      }
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  if (KM % 4 == 0 && K == KM && ((size_t)w & 15) == 0) {     // a channel's taps by fours: one by one, each load touches every line
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        const int d = min((c * 64 + lane) * VE + e, nd - 1);
#pragma unroll
        for (int k = 0; k < KM; k += 4) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(w + (long)(col + d) * KM + k);
#pragma unroll
          for (int i = 0; i < 4; ++i) wk[k + i][c * VE + e] = v[i];
        }
      }
  } else {
#pragma unroll
    for (int k = 0; k < KM; ++k)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < VE; ++e) {
          const int d = (c * 64 + lane) * VE + e;
          wk[k][c * VE + e] = (d < nd && k >= pad) ? w[(long)(col + d) * K + k - pad] : 0.f;
        }
  }
  // the slot's next history: entry e is the input K-1-e rows before the segment's end (entries move down, so each
  // is read before it is overwritten; a lane touches its own channels only)
  if (keep) {
#pragma unroll
    for (int e = 0; e < (KM <= 8 ? KM - 1 : 0); ++e)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int d = (c * 64 + lane) * VE;
        if (d < nd && e < K - 1) {
#pragma unroll
          for (int q = 0; q < VE; ++q) st[(long)e * C + d + q] = h[e][c * VE + q];
        }
      }
    for (int e = 0; KM > 8 && e < K - 1; ++e) {
      const int i = n - (K - 1) + e;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int d = (c * 64 + lane) * VE;
        if (d < nd) {
#pragma unroll
          for (int q = 0; q < VE; ++q)
            st[(long)e * C + d + q] = i >= 0 ? ldf(in + (long)(r0 + i) * si + col + d + q)
                                             : (fresh ? 0.f : st[(long)(e + n) * C + d + q]);
        }
      }
    }
  }
  float nw[NV];
  const float* wn = isq ? qw : (isv ? nullptr : kw);
  if (wn != nullptr)
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        const int d = (c * 64 + lane) * VE + e;
        nw[c * VE + e] = d < nd ? wn[d] : 0.f;
      }
  const int Wr = G * (D + P);
  // four rows at a time, so that their reductions run side by side
#pragma unroll
  for (int i0 = 0; i0 < TT; i0 += RB) {
    if (t0 + i0 >= n) break;
    float y[RB][NV], ss[RB];
    int at[RB];                                           // position of a query, cache row of a key or value
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const long row = r0 + min(t0 + i0 + i, n - 1);
      at[i] = isq ? (tcoef != 0.f ? pos[row] : 0) : slots[row];
      ss[i] = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        float a = 0.f;
#pragma unroll
        for (int k = 0; k < KM; ++k) a += wk[k][v] * x[i0 + i + k][v];
        y[i][v] = a;
        ss[i] += a * a;
      }
    }
    if (wn != nullptr) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int i = 0; i < RB; ++i) ss[i] += __shfl_xor(ss[i], o, 64);
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const float f = 1.0f / sqrtf(ss[i] / (float)nd + eps);
#pragma unroll
        for (int v = 0; v < NV; ++v) y[i][v] *= f * nw[v];
      }
    }
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      if (t0 + i0 + i >= n) break;
      const long row = r0 + t0 + i0 + i;
      T* dst;
      if (isq) {
        if (tcoef != 0.f) {
          const float f = 1.0f + tcoef * logf((float)((at[i] + 1) / tevery + 1));
#pragma unroll
          for (int v = 0; v < NV; ++v) y[i][v] *= f;
        }
        dst = qout + row * (long)H * D + (long)unit * D;
      } else {
        if (at[i] < 0) continue;
        dst = cache + (long)at[i] * Wr + (isv ? G * D + (unit - H - G) * P : (unit - H) * D);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int d = (c * 64 + lane) * VE;
        if (d < nd) {
          vt o;
#pragma unroll
          for (int e = 0; e < VE; ++e) o[e] = (T)y[i][c * VE + e];
          *reinterpret_cast<vt*>(dst + d) = o;
        }
      }
    }
  }
}

}  // namespace

// in: [T, C] slice (row stride si) of storage type dt, channels q: H*D | k: G*D | v: G*P; w f32 [C, K] (last column:
// the current token's tap), 1 <= K <= 16; state f32 [slots, K-1, C] (unused for K = 1); qw / kw f32 [D] or null;
// cu [S+1] row bounds, slot [S] (< 0: no history kept), pos [T], slots [T] cache rows (< 0: no write);
// cache [rows, G*(D+P)] (unused for G = 0) and qout [T, H*D] of storage type dt
MX_API int mx_conv_heads(const void* in, long si, int dt, const float* w, int K, float* state, const float* qw,
                         const float* kw, float eps, float tcoef, int tevery, const int* cu, const int* slot,
                         const int* pos, const int* slots, void* cache, void* qout, int S, int max_len, int rows, int H, int G,
                         int D, int P, hipStream_t st) {
  if (S <= 0 || max_len <= 0) return 0;
  const int big = G > 0 && P > D ? P : D;
  if (K < 1 || K > 16 || H < 1 || G < 0 || D < 1 || P < 1 || big > 512 || tevery < 1 || (K > 1 && state == nullptr) ||
      (G > 0 && cache == nullptr))
    return (int)hipErrorInvalidValue;
  const size_t al = dt == 1 ? 8 : 4;                       // two elements
  const bool two = D % 2 == 0 && (G == 0 || P % 2 == 0) && si % 2 == 0 && ((size_t)in | (size_t)qout | (size_t)cache) % al == 0;
  const int units = H + 2 * G;
  // Rows per wave: a wave's rows follow each other's loads, so that few are the shorter way until memory is the bound (bf16, 16 query heads
  // over 4, four taps, us, before with 8 rows one after the other / by the rule: 100 rows 10.2 / 5.9, 400 11.2 / 6.3, 1160 15.2 /
  // 11.9, 2048 20.2 / 15.0, 4096 29.7 / 26.1, 40 single rows 5.6 / 4.3; of these, the taps by fours were 8.2, 8.8, 14.4, 17.6, 31.4 and 5.6 before).
  // A wave of 8 or 16 rows fetches as many for a segment of one: five taps, 1, 64 and 200 single rows, with 8 rows one after the other / by 8
  // side by side / by one 5.4 / 6.2 / 5.0, 6.8 / 7.6 / 6.2, 10.9 / 11.8 / 10.0.
#define CH_LAUNCH(VE, NC, KM, TT)                                                                                     \
  do {                                                                                                                \
    dim3 grid(mx_tile_count(S, rows, max_len, TT, 6), (units + CH_WAVES - 1) / CH_WAVES);                             \
    MX_DISPATCH(dt, TY, conv_heads_kernel<TY, VE, NC, KM, TT><<<grid, CH_WAVES * 64, 0, st>>>(                        \
        (const TY*)in, si, w, K, state, qw, kw, eps, tcoef, tevery, cu, slot, pos, slots, (TY*)cache, (TY*)qout,       \
        S, mx_tile_per(S, rows, max_len, TT, 6), H, G, D, P));                                                         \
  } while (0)
#define CH_TAPS(VE, NC)                     \
  do {                                      \
    if (K <= 4 && max_len == 1) CH_LAUNCH(VE, NC, 4, 1); \
    else if (K <= 4 && rows * (long)units < 24000) CH_LAUNCH(VE, NC, 4, 4); \
    else if (K <= 4) CH_LAUNCH(VE, NC, 4, 8); \
    else if (K <= 8 && max_len == 1) CH_LAUNCH(VE, NC, 8, 1); \
    else if (K <= 8) CH_LAUNCH(VE, NC, 8, 8); \
    else if (max_len == 1) CH_LAUNCH(VE, NC, 16, 1); \
    else CH_LAUNCH(VE, NC, 16, 16);         \
  } while (0)
  if (two) {
    if (big <= 128) CH_TAPS(2, 1);
    else if (big <= 256) CH_TAPS(2, 2);
    else CH_TAPS(2, 4);
  } else {
    if (big <= 128) CH_TAPS(1, 2);
    else CH_TAPS(1, 8);
  }
#undef CH_TAPS
#undef CH_LAUNCH
  MX_RETURN_LAUNCH();
}
