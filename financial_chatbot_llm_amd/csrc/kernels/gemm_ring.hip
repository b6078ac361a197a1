// Projections of 257 to 3072 rows (prompts):
//   Y[m, n] = sum_k X[m, k] * W[n, k]          X [M, K] bf16 (row stride ldx), W [N, K] bf16 row-major, Y [M, N] bf16
//
// At these sizes a product is one round of blocks over the 256 CUs, and what counts is that the round is well filled and that a
// block's chain of K steps never waits for memory.  So: ten tiles, from 64 x 64 to 256 x 160, of which penny_linear_ring_plan takes
// the one whose single round is the shortest; one block of eight waves per CU; and as many stages of K as LDS holds (3 to 6, 140 -
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
// Epilogues: the rounded product; the residual stream added to it; f32 slabs of S slices of K, which the consumer adds; and of a QKV
// projection (heads of 128) rotation and the paged cache's layout, each with the roundings of gemm_prefill.hip's.  For the last a
// wave's W rows are 32 of a head's first half and the 32 that they turn with, so that both meet in one lane.
#include "common.h"
#include "kv_layout.h"

#include <cfloat>

extern "C" float penny_linear_rows_us(int M, int N, int K);

namespace {

union Frag {
  uint4 u;
  bf16x8 v;
};

template <int N_>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_) : "memory");
}

enum { RING_PLAIN, RING_RESIDUAL, RING_ROPE, RING_SLABS };

struct RingRope {
  const int* positions;   // [M]
  const float* cos_sin;   // [max_pos, 128]: cos of the 64 frequencies, then sin
  const int* slots;       // [M] slot in the paged cache, < 0: not stored
  bf16* q;                // [M, Hq, 128]
  bf16* k_cache;
  bf16* v_cache;
  int Hq, Hkv;
  float qscale;           // on the rotated q before its rounding
};

template <int TN, int TM, int KG, int NST, int EPI>
__global__ void __launch_bounds__(512) linear_ring_kernel(const char* __restrict__ X, int ldx, const char* __restrict__ W, int K,
                                                          bf16* Y, int ldy, const bf16* R, int ldr, int M, int N, int S,
                                                          RingRope rope) {
  constexpr int WN = TN / 64, WM = 8 / (KG * WN), UF = TM / WM / 16;      // waves over W rows, over tokens; token groups of a wave
  constexpr int ROWB = KG == 1 ? 128 : 64 * KG, CPR = ROWB / 16, RPP = 1024 / ROWB;
  constexpr int STG = (TN + TM) * ROWB, PIECES = STG / 1024, LPS = (PIECES + 7) / 8, WP = TN * ROWB / 1024;
  static_assert(NST * STG <= 163840 && 2 * UF % KG == 0 && (NST - 1) * LPS < 64, "LDS, shares of the sum, the wait's counter");
  static_assert(KG == 1 || 8 * 4 * UF / KG * 1024 <= NST * STG, "the groups' sums meet in the ring");
  __shared__ __attribute__((aligned(1024))) char smem[NST * STG];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = w % KG, pos = w / KG, wa = pos / WM, wb = pos % WM, g = lane >> 4, col = lane & 15;

  const int Mt = (M + TM - 1) / TM, Nt = (N + TN - 1) / TN, nwg = Mt * Nt * S;
  int id = blockIdx.x;
  {
    const int xcd = id & 7, q = nwg >> 3, r = nwg & 7;
    id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (id >> 3);
  }
  const int slice = EPI == RING_SLABS ? id / (Mt * Nt) : 0;
  if (EPI == RING_SLABS) id -= slice * (Mt * Nt);
  const int grp = id / (8 * Nt), first = grp * 8, gm = min(Mt - first, 8), within = id - grp * 8 * Nt;
  const int m0 = (first + within % gm) * TM, n0 = (within / gm) * TN;
  const int nt = K / S * 2 / ROWB;
  PENNY_DASSERT(nt >= 1 && nt * S * ROWB == K * 2 && m0 < M && n0 < N && slice < S);
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
  const char* wk = W + (long)slice * nt * ROWB;
  const char* xk = X + (long)slice * nt * ROWB;
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
  const char* wrd = smem + ((EPI == RING_ROPE ? (wa >> 1) * 128 + (wa & 1) * 32 : wa * 64) + col) * ROWB;
  auto frow = [](int f) { return EPI == RING_ROPE ? (f & 1) * 16 + (f >> 1) * 64 : f * 16; };
  const char* xrd = smem + (TN + wb * 16 * UF + col) * ROWB;
  int rbuf = 0;
  auto read = [&](Operands& o, int ch) {
#pragma unroll
    for (int f = 0; f < 4; ++f) o.a[f].u = *reinterpret_cast<const uint4*>(wrd + rbuf + frow(f) * ROWB + ch);
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

  // item i of a wave's 2 UF: two of its row groups (neighbours, or those that turn together) of its tokens 16 (i / 2) .. + 15; of KG
  // waves the kg-th adds up and writes the items kg IW ..
  constexpr int IW = 2 * UF / KG;
  auto fa = [](int i) { return EPI == RING_ROPE ? i & 1 : 2 * (i & 1); };
  auto fb = [&](int i) { return fa(i) + (EPI == RING_ROPE ? 2 : 1); };
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
            sums[i * 128] = acc[fa(i)][i >> 1];
            sums[i * 128 + 64] = acc[fb(i)][i >> 1];
          }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < KG; ++j)
        if (kg == j)
#pragma unroll
          for (int i = j * IW; i < (j + 1) * IW; ++i) {
            acc[fa(i)][i >> 1] += sums[i * 128];
            acc[fb(i)][i >> 1] += sums[i * 128 + 64];
          }
    }
  }
  const int n = n0 + wa * 64 + 8 * (g >> 1) + 16 * (g & 1);
#pragma unroll
  for (int j = 0; j < KG; ++j) {
    if (kg != j) continue;
#pragma unroll
    for (int i = j * IW; i < (j + 1) * IW; ++i) {
      const int u = i >> 1, m = m0 + (wb * UF + u) * 16 + col;
      if (m >= M) continue;               // all four lanes of a token row together: their swaps have partners
      const f32x4 ca = acc[fa(i)][u], cb = acc[fb(i)][u];
      if constexpr (EPI == RING_SLABS) {
        const int c = n0 + wa * 64 + 16 * fa(i) + 4 * g;
        float* P = reinterpret_cast<float*>(Y) + ((long)slice * M + m) * N + c;
        if (c < N) *reinterpret_cast<f32x4*>(P) = ca;
        if (c + 16 < N) *reinterpret_cast<f32x4*>(P + 16) = cb;
        continue;
      }
      bf16x4 lo, hi;
#pragma unroll
      for (int r = 0; r < 4; ++r) lo[r] = (bf16)ca[r], hi[r] = (bf16)cb[r];
      if constexpr (EPI == RING_ROPE) {
        const int hd = (n0 >> 7) + (wa >> 1), d = (wa & 1) * 32 + 16 * (i & 1) + 4 * g, slot = rope.slots[m];
        if (hd >= rope.Hq + 2 * rope.Hkv || (hd >= rope.Hq && slot < 0)) continue;
        const long blk = slot >= 0 ? slot / KV_BS : 0;
        const int at = slot >= 0 ? slot % KV_BS : 0;
        if (hd < rope.Hq + rope.Hkv) {
          const float* cs = rope.cos_sin + (long)rope.positions[m] * 128 + d;
          const f32x4 co = *reinterpret_cast<const f32x4*>(cs), si = *reinterpret_cast<const f32x4*>(cs + 64);
          const float qs = hd < rope.Hq ? rope.qscale : 1.f;
          bf16x4 o1, o2;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float x1 = (float)lo[r], x2 = (float)hi[r];
            o1[r] = (bf16)((x1 * co[r] - x2 * si[r]) * qs);
            o2[r] = (bf16)((x2 * co[r] + x1 * si[r]) * qs);
          }
          if (hd < rope.Hq) {
            bf16* q = rope.q + ((long)m * rope.Hq + hd) * 128 + d;
            *reinterpret_cast<bf16x4*>(q) = o1;
            *reinterpret_cast<bf16x4*>(q + 64) = o2;
          } else {
            bf16* kb = rope.k_cache + (blk * rope.Hkv + (hd - rope.Hq)) * (long)(KV_BS * 128);
            *reinterpret_cast<bf16x4*>(kb + k_index(at, d, 128)) = o1;
            *reinterpret_cast<bf16x4*>(kb + k_index(at, 64 + d, 128)) = o2;
          }
        } else {
          bf16* vb = rope.v_cache + (blk * rope.Hkv + (hd - rope.Hq - rope.Hkv)) * (long)(KV_BS * 128);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            vb[v_index(at, d + r, 128)] = lo[r];
            vb[v_index(at, 64 + d + r, 128)] = hi[r];
          }
        }
      } else {
        const int c = n + 16 * fa(i);
        Pack8 v;
        v.u = pair16(lo, hi);
        if (c >= N) continue;
        if constexpr (EPI == RING_RESIDUAL) {   // rounded as the product and the addition one after the other
          Pack8 r;
          r.u = *reinterpret_cast<const uint4*>(R + (long)m * ldr + c);
#pragma unroll
          for (int e = 0; e < 8; ++e) v.e[e] = (bf16)((float)v.e[e] + (float)r.e[e]);
        }
        *reinterpret_cast<uint4*>(Y + (long)m * ldy + c) = v.u;
      }
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
static int ring_plan(int M, int N, int K, int narrowest, float& best, int S = 1) {
  int plan = 0;
  for (int i = 0; i < kRingCount; ++i) {
    const RingTile& t = kRingTiles[i];
    if (t.tn < narrowest || K % ((t.kg == 1 ? 64 : 32 * t.kg) * S) || ring_blocks(t, M, N) * S > 256) continue;
    const float us = t.fixed + t.step * K / S / 64;
    if (us < best) best = us, plan = i + 1;
  }
  return plan;
}
PENNY_API int penny_linear_ring_plan(int M, int N, int K) {
  if (M <= 256 || M > 3072 || N < 512 || N % 8 || (N > 8192 && M > 384) || K <= 0 || K % 64) return 0;
  float us = penny_linear_rows_us(M, N, K);
  return ring_plan(M, N, K, 0, us);
}
// The same for products that the library does otherwise (ops.gemm.project), or 0.  Where W's rows are in whole 256s the library's large tiles
// have no remainder, and from 128 x 256 on the ring's are slower (weights beyond the caches, library / here: 4096 x 2048, 1600 rows 33.9 / 37.9, 2557
// 44.3 / 47.2; 5120 x 2048, 1200 - 1450 rows 0.94 of its rate, 1724 0.91; 2560 x 1024, 2400 - 3000 rows 0.97; 4096 x 6144, 2557 rows 111.6 / 119.4; a few
// sizes that the library does badly are faster here: 6144 x 1024, 1458 rows 1.26); beside other widths they are the faster at all sizes (5168 x 2048 1.03 -
// 1.10, 3592 x 1024 1.09 - 1.26).
PENNY_API int penny_project_ring_plan(int M, int N, int K) {
  const int tile = penny_linear_ring_plan(M, N, K);
  return tile && N % 256 == 0 && K >= 1024 && kRingTiles[tile - 1].tn * kRingTiles[tile - 1].tm >= 128 * 256 ? 0 : tile;
}
// The tile of penny_qkv_ring for heads of 128, or 0: the 256 x 256 tiles of gemm_prefill.hip are left what no single round holds
// (6144 x 4096 with rotation and scattered cache rows, us there / here: 300 rows 73 / 37, 476 77 / 48, 768 90 / 66, 1176 114 / 94, 1600 115 /
// 107; 10240 x 8192 374 rows 118 / 89, 900 198 / 176)
PENNY_API int penny_qkv_ring_plan(int M, int N, int K) {
  if (M <= 256 || M > 3072 || N <= 0 || N % 128 || K <= 0 || K % 64) return 0;
  float us = FLT_MAX;
  return ring_plan(M, N, K, 128, us);
}
// The tile of penny_ring_slabs for S slices, or 0: no single round holds them.  With the norm that adds the slabs, us on gemm_mid.hip's
// 128 x 128 tiles / here: 4096 x 14336 in 4 slices 260 rows 65 / 52, 374 69 / 59, 512 85 / 74; 4096 x 4096 in 4 300 rows 28.7 / 25.1, in 2 640 rows
// 40.7 / 34.7; 1280 x 8192 in 8 448 rows 27.4 / 23.8, 896 40.9 / 36.1.  (Beside 256 x 256 tiles in slices it is level at 640 rows and slower
// from there: 4096 x 14336, 1024 rows 107 / 119.)
PENNY_API int penny_ring_slabs_plan(int M, int N, int K, int S) {
  if (M <= 256 || M > 3072 || N < 512 || N % 8 || K <= 0 || K % 64 || S < 1 || S > 64) return 0;
  float us = FLT_MAX;
  return ring_plan(M, N, K, 0, us, S);
}

// one line per entry of kRingTiles; the first two have too few W rows for a head
#define RING_TILES_WIDE(F)                                                                                          \
  F(3, 128, 64, 2, 6) F(4, 128, 96, 2, 5) F(5, 128, 128, 2, 5) F(6, 128, 160, 2, 4) F(7, 128, 192, 2, 4) F(8, 128, 256, 2, 3) \
  F(9, 256, 128, 1, 3) F(10, 256, 160, 1, 3)
#define RING_TILES(F) F(1, 64, 64, 4, 5) F(2, 64, 128, 4, 3) RING_TILES_WIDE(F)
#define RING_LAUNCH(I, TN, TM, KG, NST, EPI, ROPE)                                                                   \
  do {                                                                                                               \
    constexpr RingTile e = kRingTiles[I - 1];                                                                        \
    static_assert(e.tn == TN && e.tm == TM && e.kg == KG && e.stages == NST, "the kernel of this entry");            \
    linear_ring_kernel<TN, TM, KG, NST, EPI><<<(unsigned)blocks, 512, 0, st>>>((const char*)X, ldx, (const char*)W, K, (bf16*)Y, ldy, \
                                                                               (const bf16*)R, ldr, M, N, S, ROPE);  \
  } while (0)

// Y [M, N] (row stride ldy) = X W^T (+ R, row stride ldr, which may be Y) on tile number `tile` (penny_linear_ring_plan).  Contract
// (checked): all rows in whole 16 bytes, N a multiple of 8, K of 64 and of the tile's step, each operand below 4 GiB.
PENNY_API int penny_linear_ring(const void* X, int ldx, const void* W, int K, void* Y, int ldy, const void* R, int ldr, int M, int N,
                                int tile, hipStream_t st) {
  if (M <= 0) return 0;
  if (tile < 1 || tile > kRingCount || N <= 0 || N % 8 || K <= 0 || K % 64 || ldx < K || ldx % 8 || ldy < N || ldy % 8 ||
      (R != nullptr && (ldr < N || ldr % 8)) || ((size_t)X | (size_t)W | (size_t)Y | (size_t)R) % 16 || (long)M * ldx >= 1L << 31 ||
      (long)N * K >= 1L << 31)
    return (int)hipErrorInvalidValue;
  const RingTile& t = kRingTiles[tile - 1];
  const int S = 1;
  const long blocks = ring_blocks(t, M, N);
  if (K % (32 * t.kg) || blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
#define RING(I, TN, TM, KG, NST)                                                                                  \
  case I:                                                                                                         \
    if (R != nullptr) RING_LAUNCH(I, TN, TM, KG, NST, RING_RESIDUAL, RingRope{});                                 \
    else RING_LAUNCH(I, TN, TM, KG, NST, RING_PLAIN, RingRope{});                                                 \
    break;
  switch (tile) { RING_TILES(RING) }
#undef RING
  PENNY_RETURN_LAUNCH();
}

// The QKV projection of penny_gemm_prefill_qkv_rope on tile number `tile` (penny_qkv_ring_plan): q [M, Hq, 128] rotated and times qscale, k and
// v scattered into the paged caches.  Contract (checked) as above.
PENNY_API int penny_qkv_ring(const void* X, int ldx, const void* W, int K, int M, const int* positions, const float* cos_sin, const int* slots,
                             void* q_out, void* k_cache, void* v_cache, int Hq, int Hkv, float qscale, int tile, hipStream_t st) {
  if (M <= 0) return 0;
  const int N = (Hq + 2 * Hkv) * 128, ldy = 0, ldr = 0;
  void* Y = nullptr;
  const void* R = nullptr;
  if (tile < 3 || tile > kRingCount || Hq <= 0 || Hkv <= 0 || Hq + 2L * Hkv > 1 << 20 || K <= 0 || K % 64 || ldx < K || ldx % 8 || !positions ||
      !cos_sin || !slots || !q_out || !k_cache || !v_cache || ((size_t)X | (size_t)W | (size_t)cos_sin) % 16 ||
      ((size_t)q_out | (size_t)k_cache | (size_t)v_cache) % 8 || (long)M * ldx >= 1L << 31 || (long)N * K >= 1L << 31)
    return (int)hipErrorInvalidValue;
  const RingTile& t = kRingTiles[tile - 1];
  const int S = 1;
  const long blocks = ring_blocks(t, M, N);
  if (K % (32 * t.kg) || blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
  const RingRope rope{positions, cos_sin, slots, (bf16*)q_out, (bf16*)k_cache, (bf16*)v_cache, Hq, Hkv, qscale};
#define QKV(I, TN, TM, KG, NST)                               \
  case I:                                                     \
    RING_LAUNCH(I, TN, TM, KG, NST, RING_ROPE, rope);         \
    break;
  switch (tile) { RING_TILES_WIDE(QKV) }
#undef QKV
  PENNY_RETURN_LAUNCH();
}

// f32 slabs P [S, M, N] of X W^T in S slices of K on tile number `tile` (penny_ring_slabs_plan).  Contract (checked) as above, K also a
// multiple of S steps.
PENNY_API int penny_ring_slabs(const void* X, int ldx, const void* W, int K, float* P, int M, int N, int S, int tile, hipStream_t st) {
  if (M <= 0) return 0;
  void* Y = P;
  const void* R = nullptr;
  const int ldy = N, ldr = 0;
  if (tile < 1 || tile > kRingCount || S < 1 || S > 64 || N <= 0 || N % 8 || K <= 0 || K % 64 || ldx < K || ldx % 8 ||
      ((size_t)X | (size_t)W | (size_t)P) % 16 || (long)M * ldx >= 1L << 31 || (long)N * K >= 1L << 31)
    return (int)hipErrorInvalidValue;
  const RingTile& t = kRingTiles[tile - 1];
  const long blocks = ring_blocks(t, M, N) * S;
  if (K % ((t.kg == 1 ? 64 : 32 * t.kg) * S) || blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
#define SLABS(I, TN, TM, KG, NST)                                    \
  case I:                                                            \
    RING_LAUNCH(I, TN, TM, KG, NST, RING_SLABS, RingRope{});         \
    break;
  switch (tile) { RING_TILES(SLABS) }
#undef SLABS
  PENNY_RETURN_LAUNCH();
}
