// Projections of some hundred to three thousand rows (prompts of the layered decoders):
//   Y[m, n] = sum_k X[m, k] * W[n, k]          X [M, K] bf16 (row stride ldx), W [N, K] bf16 row-major, Y [M, N] bf16
//
// At these sizes a product is one round of blocks over the 256 CUs, and what counts is that the round is well filled and that a
// block's chain of K steps never waits for memory.  So: ten tiles, from 64 x 64 to 256 x 160, of which penny_linear_ring_plan takes
// the one whose single round is the shortest; one block of eight waves per CU; and as many stages of K as LDS holds (2 to 6, 96 -
// 160 KB) in flight by LDS-DMA, with counted waits.
//   * A wave's sub-tile is 64 W rows by a part of the tokens.  Tiles of up to 128 W rows have fewer sub-tiles than waves: KG groups
//     of waves then take every KG-th 32 of K of a stage, so that each still has a large sub-tile (operand reads from LDS are the
//     nearest bound, then the CU's 64 B per clock from the caches), and add up through LDS at the end.
//   * The operands of stage t + 1 are read while stage t is on the matrix cores: one barrier a stage, behind which stage t's
//     buffer is filled again.
//   * Rows of a stage are 64 KG bytes, 16-byte chunks swizzled by the row on the source address and the read (every 16 lanes of a
//     ds_read_b128 touch 16 distinct chunks).
//   * Token tiles go fastest within groups of eight and neighbouring tiles to the same XCD, so that its L2 holds the panels.
// Measured, weights beyond the caches, us library / here: 2048 x 2048 400 rows 10.9 / 10.0, 1188 19.5 / 17.2, 2600 29.7 / 25.1;
// 2048 x 6144 800 rows 39.0 / 33.8; 4096 x 2048 800 rows 24.3 / 20.9; 7216 x 2048 400 rows 25.2 / 19.9, 1188 41.9 / 39.3; 1024 x 1024 1000
// rows 9.6 / 7.4; 3592 x 1024 1500 rows 20.3 / 16.4.  A stage of 128 x 128 takes 0.48 us: LDS is busy for 0.32 of it, the matrix
// cores for 0.21.
#include "common.h"

#include <cfloat>

extern "C" float penny_linear_rows_us(int M, int N, int K);

namespace {

union Frag {
  uint4 u;
  bf16x8 v;
};

// lo = columns 16f + 4g .. +3 and hi = 16(f+1) + 4g .. +3 of lane row g -> 8 consecutive columns 8*(g>>1) + 16*(g&1) .. +7 of this lane
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

template <int N_>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_) : "memory");
}

template <int TN, int TM, int KG, int NST>
__global__ void __launch_bounds__(512) linear_ring_kernel(const char* __restrict__ X, int ldx, const char* __restrict__ W, int K,
                                                          bf16* __restrict__ Y, int M, int N) {
  constexpr int WN = TN / 64, WM = 8 / (KG * WN), UF = TM / WM / 16;      // waves over W rows, over tokens; token groups of a wave
  constexpr int ROWB = KG == 1 ? 128 : 64 * KG, CPR = ROWB / 16, RPP = 1024 / ROWB;
  constexpr int STG = (TN + TM) * ROWB, PIECES = STG / 1024, LPS = (PIECES + 7) / 8, WP = TN * ROWB / 1024;
  static_assert(NST * STG <= 163840 && 2 * UF % KG == 0 && (NST - 1) * LPS < 64, "LDS, shares of the sum, the wait's counter");
  static_assert(KG == 1 || 8 * 4 * UF / KG * 1024 <= NST * STG, "the groups' sums meet in the ring");
  __shared__ __attribute__((aligned(1024))) char smem[NST * STG];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = w % KG, pos = w / KG, wa = pos / WM, wb = pos % WM, g = lane >> 4, col = lane & 15;

  const int Mt = (M + TM - 1) / TM, Nt = (N + TN - 1) / TN, nwg = Mt * Nt;
  int id = blockIdx.x;
  {
    const int xcd = id & 7, q = nwg >> 3, r = nwg & 7;
    id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (id >> 3);
  }
  const int grp = id / (8 * Nt), first = grp * 8, gm = min(Mt - first, 8), within = id - grp * 8 * Nt;
  const int m0 = (first + within % gm) * TM, n0 = (within / gm) * TN;
  const int nt = K * 2 / ROWB;
  PENNY_DASSERT(nt >= 1 && K * 2 % ROWB == 0 && m0 < M && n0 < N);
  auto swz = [](int r) { return CPR == 8 ? (r >> 1) & 7 : r & 15; };

  // this wave's 1-KiB pieces of a stage: W rows, then tokens; rows beyond the operands and pieces beyond the stage are read twice
  unsigned off[LPS];
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const int p = min(w + 8 * i, PIECES - 1), r = p * RPP + lane / CPR, c = (lane % CPR) ^ swz(r);
    const bool isw = p < WP;
    const int row = isw ? min(n0 + r, N - 1) : min(m0 + r - TN, M - 1);
    off[i] = (unsigned)row * (unsigned)((isw ? K : ldx) * 2) + 16 * c;
  }
  const unsigned lds0 = (unsigned)(uintptr_t)((__attribute__((address_space(3))) char*)smem);
  const char* wk = W;
  const char* xk = X;
  unsigned sbuf = lds0;
  // inline-asm DMA: hipcc does not see it, so the operand reads are not held behind it; the counted waits below are the only ones
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < LPS; ++i) {
      const int p = min(w + 8 * i, PIECES - 1);
      const char* base = p < WP ? wk : xk;
      unsigned keep;
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep)
                   : "v"(off[i]), "s"(sbuf + p * 1024), "s"(base)
                   : "memory");
    }
    wk += ROWB;
    xk += ROWB;
    sbuf = sbuf + STG == lds0 + NST * STG ? lds0 : sbuf + STG;
  };
  auto wait_stage = [&](int young) {      // until at most `young` newer stages are in flight
    if (young >= NST - 2) wait_vm<(NST - 2) * LPS>();
    else if (NST > 5 && young == 3) wait_vm<3 * LPS>();
    else if (NST > 4 && young == 2) wait_vm<2 * LPS>();
    else if (NST > 3 && young == 1) wait_vm<LPS>();
    else wait_vm<0>();
  };

  struct Operands {
    Frag a[4], b[UF];
  };
  const int ch0 = ((KG > 1 ? 4 * kg + g : g) ^ swz(col)) << 4, ch1 = ((4 + g) ^ swz(col)) << 4;
  const char* wrd = smem + (wa * 64 + col) * ROWB;
  const char* xrd = smem + (TN + wb * 16 * UF + col) * ROWB;
  int rbuf = 0;
  auto read = [&](Operands& o, int ch) {
#pragma unroll
    for (int f = 0; f < 4; ++f) o.a[f].u = *reinterpret_cast<const uint4*>(wrd + rbuf + f * 16 * ROWB + ch);
#pragma unroll
    for (int u = 0; u < UF; ++u) o.b[u].u = *reinterpret_cast<const uint4*>(xrd + rbuf + u * 16 * ROWB + ch);
  };
  f32x4 acc[4][UF];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int u = 0; u < UF; ++u) acc[f][u] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Operands& o) {
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int u = 0; u < UF; ++u) acc[f][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.a[f].v, o.b[u].v, acc[f][u], 0, 0, 0);
  };
  // stage t has been read by this wave (lgkmcnt) and t + 1 has landed; behind the barrier both hold for all waves
  auto advance = [&](int t, Operands& o) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    wait_stage(min(nt, t + NST) - (t + 2));
    __builtin_amdgcn_s_barrier();
    rbuf = rbuf + STG == NST * STG ? 0 : rbuf + STG;
    read(o, ch0);
    if (t + NST < nt) stage();
  };

  const int ahead = min(nt, NST);
  for (int t = 0; t < ahead; ++t) stage();
  if (nt >= NST) wait_vm<(NST - 1) * LPS>();
  else wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  Operands p, q;
  read(p, ch0);
  if constexpr (KG > 1) {                 // a stage is one step of 32 of K for every group
    int t = 0;
    for (; t + 1 < nt; t += 2) {
      advance(t, q);
      multiply(p);
      if (t + 2 < nt) advance(t + 1, p);
      multiply(q);
    }
    if (t < nt) multiply(p);
  } else {
    for (int t = 0; t < nt; ++t) {
      read(q, ch1);
      multiply(p);
      if (t + 1 < nt) advance(t, p);
      multiply(q);
    }
  }

  // item i of a wave's 2 UF: columns 32 (i % 2) .. + 31 of its tokens 16 (i / 2) .. + 15; of KG waves the kg-th adds up and
  // writes the items kg IW ..
  constexpr int IW = 2 * UF / KG;
  if constexpr (KG > 1) {
    f32x4* sums = reinterpret_cast<f32x4*>(smem) + pos * KG * (IW * 128) + lane;
#pragma unroll
    for (int r = 1; r < KG; ++r) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < KG; ++j)
        if ((kg + r) % KG == j)
#pragma unroll
          for (int i = j * IW; i < (j + 1) * IW; ++i) {
            sums[i * 128] = acc[2 * (i & 1)][i >> 1];
            sums[i * 128 + 64] = acc[2 * (i & 1) + 1][i >> 1];
          }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < KG; ++j)
        if (kg == j)
#pragma unroll
          for (int i = j * IW; i < (j + 1) * IW; ++i) {
            acc[2 * (i & 1)][i >> 1] += sums[i * 128];
            acc[2 * (i & 1) + 1][i >> 1] += sums[i * 128 + 64];
          }
    }
  }
  const int n = n0 + wa * 64 + 8 * (g >> 1) + 16 * (g & 1);
#pragma unroll
  for (int j = 0; j < KG; ++j) {
    if (kg != j) continue;
#pragma unroll
    for (int i = j * IW; i < (j + 1) * IW; ++i) {
      const int f = 2 * (i & 1), u = i >> 1, m = m0 + (wb * UF + u) * 16 + col;
      if (m >= M) continue;               // all four lanes of a token row together: their swaps have partners
      bf16x4 lo, hi;
#pragma unroll
      for (int r = 0; r < 4; ++r) lo[r] = (bf16)acc[f][u][r], hi[r] = (bf16)acc[f + 1][u][r];
      const uint4 v = pair16(lo, hi);
      if (n + 16 * f < N) *reinterpret_cast<uint4*>(Y + (long)m * N + n + 16 * f) = v;
    }
  }
}

// The tiles (W rows, tokens, groups of K, stages) with what a block takes: us per 64 of K and beside that, fitted to single rounds of
// more than 128 blocks (200 products of 300 - 5065 rows: the choice by them is within 0.3 % of the best tile)
struct RingTile {
  int tn, tm, kg, stages;
  float step, fixed;
};
constexpr RingTile kRingTiles[] = {{64, 64, 4, 5, 0.243f, 3.0f},   {64, 128, 4, 3, 0.344f, 3.8f},  {128, 64, 2, 6, 0.402f, 2.6f},
                                   {128, 96, 2, 5, 0.450f, 3.8f},  {128, 128, 2, 5, 0.484f, 5.0f}, {128, 160, 2, 4, 0.541f, 6.0f},
                                   {128, 192, 2, 4, 0.614f, 5.8f}, {128, 256, 2, 3, 0.798f, 6.5f}, {256, 128, 1, 3, 0.862f, 4.6f},
                                   {256, 160, 1, 3, 1.058f, 4.5f}};
constexpr int kRingCount = sizeof(kRingTiles) / sizeof(kRingTiles[0]);

long ring_blocks(const RingTile& t, int M, int N) { return (long)((M + t.tm - 1) / t.tm) * ((N + t.tn - 1) / t.tn); }

}  // namespace

// The tile of penny_linear_ring for these sizes, counted from 1, or 0: no tile holds them in one round of blocks, or another path is
// the faster.  Beyond one round the library's products, which share out a last part-filled one, are (7216 x 2048, 2600 rows: level;
// 4096 x 2048, 3453 rows 47.7 / 65.0), as they are for many columns (12288 x 2048, 640 rows 34.2 / 35.8, 1188 52.7 / 67.9) and from some 3000
// rows on (2048 x 6144, 5065 rows: 101.7 / 119.2); up to 256 rows, and where they are estimated to be shorter, the streaming tiles of
// penny_linear_rows.
PENNY_API int penny_linear_ring_plan(int M, int N, int K) {
  if (M <= 256 || M > 3072 || N < 512 || N % 8 || (N > 8192 && M > 384) || K <= 0 || K % 64) return 0;
  int plan = 0;
  float best = penny_linear_rows_us(M, N, K);
  for (int i = 0; i < kRingCount; ++i) {
    const RingTile& t = kRingTiles[i];
    if (K % (32 * t.kg) || ring_blocks(t, M, N) > 256) continue;
    const float us = t.fixed + t.step * K / 64;
    if (us < best) best = us, plan = i + 1;
  }
  return plan;
}

// Y [M, N] (contiguous) = X W^T on tile number `tile` (penny_linear_ring_plan).  Contract (checked): rows of X and W in whole 16 bytes, N a
// multiple of 8, K of 64 and of the tile's step, each operand below 4 GiB.
PENNY_API int penny_linear_ring(const void* X, int ldx, const void* W, int K, void* Y, int M, int N, int tile, hipStream_t st) {
  if (M <= 0) return 0;
  if (tile < 1 || tile > kRingCount || N <= 0 || N % 8 || K <= 0 || K % 64 || ldx < K || ldx % 8 ||
      ((size_t)X | (size_t)W | (size_t)Y) % 16 || (long)M * ldx >= 1L << 31 || (long)N * K >= 1L << 31)
    return (int)hipErrorInvalidValue;
  const RingTile& t = kRingTiles[tile - 1];
  const long blocks = ring_blocks(t, M, N);
  if (K % (32 * t.kg) || blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
#define RING(I, TN, TM, KG, NST)                                                                                                 \
  case I:                                                                                                                        \
    static_assert(kRingTiles[I - 1].tn == TN && kRingTiles[I - 1].tm == TM && kRingTiles[I - 1].kg == KG && kRingTiles[I - 1].stages == NST, ""); \
    linear_ring_kernel<TN, TM, KG, NST><<<(unsigned)blocks, 512, 0, st>>>((const char*)X, ldx, (const char*)W, K, (bf16*)Y, M, N); \
    break
  switch (tile) {
    RING(1, 64, 64, 4, 5);
    RING(2, 64, 128, 4, 3);
    RING(3, 128, 64, 2, 6);
    RING(4, 128, 96, 2, 5);
    RING(5, 128, 128, 2, 5);
    RING(6, 128, 160, 2, 4);
    RING(7, 128, 192, 2, 4);
    RING(8, 128, 256, 2, 3);
    RING(9, 256, 128, 1, 3);
    RING(10, 256, 160, 1, 3);
  }
#undef RING
  PENNY_RETURN_LAUNCH();
}
