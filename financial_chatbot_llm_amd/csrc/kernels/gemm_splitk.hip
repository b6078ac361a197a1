// Mid-batch decode projection GEMM (K3/K8/K10 at 32 < M <= 256 tokens): f32 split-K slabs
//   P[s, m, n] = sum_{k in slice s} X[m, k] * W[n, k]        (Y = sum_s P[s] is reduced by the consumer)
//
// Why not hipBLASLt here: at M = 64..256 the QKV / O / down projections are still weight streams
// (33-117 MB of W against <= 7 MB of X) but the library runs them at 1.7-2.6 TB/s -- its tiles
// leave most CUs idle at N = 4096-6144 or re-read X per narrow tile.  This kernel is shaped for
// the stream instead:
//   * one workgroup = 4 waves owns BN = 16*NF rows of W and one K slice (split-K over the grid, S
//     slices) so N = 4096 still launches >= 256 workgroups; slice s = blockIdx.x % S keeps each
//     XCD on 8/S K slices, so X's L2 footprint per XCD is X/S (down-proj X is 7 MB at M = 256);
//   * BOTH operands stream into LDS with global_load_lds (16 B per lane, 1-KiB lane-linear pieces):
//     W from its MFMA-fragment-tiled copy (ops/gemm.py tile_weight -- each piece IS one A
//     fragment), X in full 128-B lines (8 token rows x 64 k per piece) with an XOR-swizzled image
//     chosen on the SOURCE address so the 16-lane phases of the fragment reads are conflict-free;
//     X is fetched once per workgroup and shared by its 4 waves (X/W on-chip traffic = M/BN);
//   * NBUF-deep ring (3-8, what fits in LDS) of BK = 64 stages, counted `s_waitcnt vmcnt` + one raw s_barrier per stage (no
//     vmcnt(0) drain in the steady state, no VGPR-destination loads in the loop at all);
//   * waves split the (W rows x tokens) tile WA x WB; v_mfma_f32_16x16x32_bf16, f32 accumulate;
//   * the epilogue writes the f32 partial tile (16-B stores); no in-launch reduction -- the next
//     kernel that reads Y anyway (residual-add+RMSNorm, RoPE/KV-write, or penny_splitk_reduce)
//     sums the S slabs, which costs S*4 B per output instead of a 1.5-2 us kernel boundary.
#include "common.h"

#include <cfloat>
#include <utility>

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void gbl_void_t;

namespace {

template <int N>
__device__ __forceinline__ void vmcnt_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

union Frag {
  uint4 u;
  bf16x8 v;
  f32x4 f;
};

// epilogues of splitk_gemm_kernel
enum { SK_SLAB = 0, SK_SILU = 1, SK_BF16 = 2, SK_SAMPLE = 3, SK_F32 = 4, SK_BIAS = 5 };

// SK_SAMPLE (the streaming LM head + K12 sampler): per-row temperature (<= 0: greedy) and seed;
// pv / pi [M, pstride] partial (best score, token) per (row, workgroup tile, wave row).  Token
// ids are voff + local row; local rows >= vvalid (a vocab shard's padding) never win.
struct SkSample {
  const float* temps;
  const unsigned long long* seeds;
  float* pv;
  int* pi;
  int pstride, voff, vvalid;
  const bf16* bias;                      // SK_BIAS
  int gelu, slices;
};

// X image: token row r of a stage lives at byte r*128; its logical 16-B chunk c (k = 8c..8c+7) at
// physical chunk c ^ (r & 7) ^ ((r >> 3) & 1).  A fragment read (16 consecutive rows, one logical
// chunk) then touches 16 distinct (row parity, chunk) bank groups per 16-lane phase.
__device__ __forceinline__ int xswz(int r, int c) { return c ^ (r & 7) ^ ((r >> 3) & 1); }

// stage ring depth: as many BK=64 stages as fit in ~150 KB of LDS (one workgroup per CU), capped
// at 8 -- a CU must keep ~50-70 KB of W in flight to stream its 1/256 share of HBM bandwidth
// MAXB: ring depth cap -- 8 by default; 16 for the narrow configs (NF = 2-4 rows groups: 4-8 KiB of
// W per stage) whose 8-stage ring keeps only 28-56 KiB in flight per CU.  Also capped so the counted
// vmcnt ((NBUF - 2) * loads per stage) fits the 6-bit counter.
// BKM: BK=64 stages issued (and waited for) in pairs -- a ring slot then holds BKM stages, so each
// W row's consecutive 128-B chunks leave the CU back to back (row-major W: 256 contiguous bytes per
// row per issue instead of 128 B one stage period apart)
template <int NF, int MT, int KB = 150, int MAXB = 8, int BKM = 1>
struct Ring {
  static constexpr int SBYTES = (NF + MT) * 2 * 1024 * BKM;
  static constexpr int LOADS = (2 * NF + 2 * MT) / 4 * BKM;
  static constexpr int BY_LDS = KB * 1024 / SBYTES;
  static constexpr int BY_VM = 63 / LOADS + 2;
  static constexpr int CAP = MAXB / BKM > 3 ? MAXB / BKM : 3;
  static constexpr int NBUF = BY_LDS < CAP ? (BY_LDS < BY_VM ? BY_LDS : BY_VM) : (CAP < BY_VM ? CAP : BY_VM);
};

// compile-time loop: f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>)
template <class F, int... U>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, U...>) {
  (f(std::integral_constant<int, U>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// wait until at most `younger` stages of this wave's glds are still in flight, then barrier
template <int LOADS, int MAXY>
__device__ __forceinline__ void wait_stage(int younger) {
  if constexpr (MAXY <= 0) {
    vmcnt_barrier<0>();
  } else {
    if (younger >= MAXY) vmcnt_barrier<MAXY * LOADS>();
    else wait_stage<LOADS, MAXY - 1>(younger);
  }
}

// MFMAs of one BK=64 stage.  `base` is __restrict__ ON PURPOSE: inlined, it gives the ds_reads
// alias-scope metadata, which is what lets hipcc's waitcnt pass leave the younger stages' LDS-DMA
// in flight -- without it the pass cannot tell them apart from this stage and drains vmcnt(0)
// before the first ds_read of every stage (measured: the ring then degenerates to one stage).
// F32: the same 16 bytes are four f32 channels 4g .. 4g + 3; the j-th of each lane make one 16x16x4 product, added into a sum of its own
// (chains a quarter as long: error of K = 1024 in one slice 5.8e-7 with one sum, 2.9e-7 with four, the library 2.9 - 5.8e-7)
template <int FW, int TW, int WBYTES, bool WROW, bool F32 = false>
__device__ __forceinline__ void stage_mma(const char* __restrict__ base, f32x4 (&acc)[F32 ? 4 : 1][FW][TW], int wa, int wb,
                                          int lane, int g, int col) {
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    Frag wf[FW], xf[TW];
#pragma unroll
    for (int f = 0; f < FW; ++f) {
      if constexpr (WROW) {   // row-major W staged like X: row r at r*128, swizzled 16-B chunks
        const int r = (wa * FW + f) * 16 + col;
        wf[f].u = *reinterpret_cast<const uint4*>(base + r * 128 + xswz(r, 4 * kk + g) * 16);
      } else {
        wf[f].u = *reinterpret_cast<const uint4*>(base + ((wa * FW + f) * 2 + kk) * 1024 + lane * 16);
      }
    }
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int r = (wb * TW + t) * 16 + col;
      xf[t].u = *reinterpret_cast<const uint4*>(base + WBYTES + r * 128 + xswz(r, 4 * kk + g) * 16);
    }
#pragma unroll
    for (int f = 0; f < FW; ++f)
#pragma unroll
      for (int t = 0; t < TW; ++t)
        if constexpr (F32) {
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j][f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[f].f[j], xf[t].f[j], acc[j][f][t], 0, 0, 0);
        } else {
          acc[0][f][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f].v, xf[t].v, acc[0][f][t], 0, 0, 0);
        }
  }
}

// Epilogues (EPI):
//   SK_BIAS   SK_BF16 with a bias row and, where asked for, the exact GELU of the rounded sum (encoder projections).  Each of
//             sa.slices slices of K is summed by itself and the slices then in turn, as by slabs: the same sums in every form;
//   SK_F32    SK_SLAB for f32 operands, which are addressed as twice as many 16-bit columns (K, ldx);
//   SK_SLAB   f32 partial slabs P [S, M, N] (reduced by the consumer's row pass);
//   SK_SILU   W is the 16-row-interleaved gate|up weight (ops/gemm.py interleave16) and S == 1: the
//             epilogue writes Y[m, f] = silu(gate) * up as bf16 [M, N/2] (ldy) instead of f32 slabs --
//             each wave owns whole (gate, up) row-group pairs, so the pair meets in one lane's registers;
//   SK_BF16   S == 1, Y bf16 [M, N] (ldy): a row-parallel TP shard whose output goes straight into the
//             all-reduce (no slab round trip, no reduce launch);
//   SK_SAMPLE S == 1, W = the [V, K] vocabulary projection (or a TP rank's padded shard): no logits
//             reach HBM -- each lane Gumbel-max-scores its bf16-rounded logits (sampler.hip's noise of
//             (row seed, global token id)) and each wave leaves one (score, token) pair per token row,
//             reduced per row by lm_sample_final_kernel (gemm_prefill.hip).  The weight-streaming LM
//             head for decode batches (M <= 128), where the 256x256 tile kernel is MFMA-bound on
//             padding rows.
// WROW: W is the plain row-major [N, K] weight (no fragment-tiled copy): its stage pieces are
// 8 rows x 128 B with the same source-side XOR swizzle as X, so every glds instruction still reads
// whole 128-B lines and the fragment reads stay conflict-free.
// RKB: LDS ring budget in KiB (150: one workgroup per CU; ~72: two co-resident workgroups, so one's
// pipeline ramp overlaps the other's stream when a CU runs several tiles in sequence).
// ONCE: the weight past the caches (nt), so that what the launches around it read -- rows, slabs, states, small weights -- stays in them.
// Its loads take longer: by itself a launch gains while its ring holds many stages (gate|up of 28672 x 4096, 16 / 32 / 64 / 128 rows, the
// weight through the caches / past them: 45.7 / 43.4, 45.5 / 42.9, 44.2 / 45.4, 53 / 61 us), but a step gains beyond that: 32 such layers
// with the tiled weight past the caches to no rows / 32 / 64 / 128: 64 rows 7504 / 7400 / 7220 / 7190 us, 96 rows 6115 / 6035 / 6015 / 5750, 128 rows
// 7330 / 7260 / 7190 / 6960; at 192 and 256 rows nothing.  Row-major weights in one chunk of rows: 8 hybrid layers of width 2048, 64 rows
// 1129 / 1078 us, 15 rows 817 / 778, 3 rows 625 / 575, f32 1 row 562 / 516, 90 rows 1231 / 1180; in several chunks, which all read the weight, 1154 and 1186
// for 100 rows.  Not for the encoder (SK_BIAS), whose weights stay on the chip from pass to pass: 60 tokens 446 and 490 us.
template <int NF, int MT, int WA, int EPI = SK_SLAB, bool WROW = false, int RKB = 150, int MAXB = 8, int BKM = 1,
          bool ONCE = !WROW && MT <= 8>
__global__ void __launch_bounds__(256, 1) splitk_gemm_kernel(const bf16* __restrict__ X, int ldx,
                                                             const bf16* __restrict__ Wt, int K,
                                                             float* __restrict__ P, int M, int N, int S,
                                                             bf16* __restrict__ Y = nullptr, int ldy = 0,
                                                             SkSample sa = SkSample{}) {
  constexpr bool SILU = EPI == SK_SILU;
  constexpr int WB = 4 / WA;
  constexpr int FW = NF / WA;   // W row groups per wave
  constexpr int TW = MT / WB;   // token tiles per wave
  static_assert(NF % WA == 0 && MT % WB == 0, "wave split");
  static_assert(!SILU || FW % 2 == 0, "SiLU epilogue needs (gate, up) row-group pairs per wave");
  constexpr int NBUF = Ring<NF, MT, RKB, MAXB, BKM>::NBUF;   // ring slots of BKM stages each
  static_assert(NBUF >= 3, "ring too shallow");
  constexpr int WBYTES = NF * 2 * 1024;        // W pieces of one BK=64 stage
  constexpr int XBYTES = MT * 2 * 1024;        // X pieces (16*MT rows x 128 B)
  constexpr int SBYTES = WBYTES + XBYTES;
  constexpr int PIECES = (2 * NF + 2 * MT);     // 1-KiB pieces per stage
  static_assert(PIECES % 4 == 0, "pieces must split evenly over 4 waves");
  constexpr int LOADS = PIECES / 4;             // glds per wave per stage
  constexpr int SLOT = BKM * SBYTES;
  __shared__ __attribute__((aligned(1024))) char smem[NBUF * SLOT];

  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, col = lane & 15;
  const int s = blockIdx.x % S, tile = blockIdx.x / S;
  // token chunks (blockIdx.y): rows m0 .. m0 + 16*MT - 1 of X / Y / the slabs; one chunk for decode
  // batches, ceil(M / (16*MT)) for the small prefill steps of narrow TP shards
  const int Mtot = M, m0 = blockIdx.y * 16 * MT;
  M = min(Mtot - m0, 16 * MT);
  X += (long)m0 * ldx;
  if constexpr (EPI == SK_SILU || EPI == SK_BF16 || EPI == SK_BIAS) Y += (long)m0 * ldy;
  PENNY_DASSERT(M > 0 && (EPI != SK_SAMPLE || gridDim.y == 1));
  PENNY_DASSERT((tile + 1) * 16 * NF <= N || (WROW && N % 8 == 0 && tile * 16 * NF < N && (EPI == SK_BF16 || EPI == SK_BIAS || EPI == SK_SLAB || EPI == SK_F32)));
  PENNY_DASSERT(K % (64 * BKM * S) == 0);
  const int n0 = tile * 16 * NF;
  const int kc = K / S, k0 = s * kc;
  const int nst = kc / (64 * BKM);              // ring slots to stream
  const int ksteps = K / 32;
  const int wa = w / WB, wb = w % WB;

  // per-lane glds source for each of this wave's pieces (fixed per kernel; advanced by k per stage)
  // piece id q = w*LOADS + i:  q < 2*NF -> W (row group q/2, k-step q%2), else X rows 8*(q-2NF)..
  const char* src[LOADS];
  int dst[LOADS];
  long step[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int q = w * LOADS + i;
    if (q < 2 * NF && WROW) {
      const int r = q * 8 + (lane >> 3);                    // weight row within the tile
      const int c = xswz(r, lane & 7);
      // the last tile of N % (16 NF) != 0 (penny_linear_rows) reads its last row again; those columns are not stored
      src[i] = reinterpret_cast<const char*>(Wt + (long)min(n0 + r, N - 1) * K + k0 + 8 * c);
      step[i] = 128;       // 64 k per stage
      dst[i] = q * 1024;
    } else if (q < 2 * NF) {
      const int f = q >> 1, kk = q & 1;
      src[i] = reinterpret_cast<const char*>(Wt) +
               (((long)(n0 / 16 + f) * ksteps + k0 / 32 + kk) * 64 + lane) * 16;
      step[i] = 2 * 1024;  // two k-steps of one row group per stage
      dst[i] = (f * 2 + kk) * 1024;
    } else {
      const int xp = q - 2 * NF;
      const int r = xp * 8 + (lane >> 3);                 // token row within the tile
      const int c = xswz(r, lane & 7);                    // logical chunk this lane's slot holds
      const int row = min(r, M - 1);
      src[i] = reinterpret_cast<const char*>(X + (long)row * ldx + k0 + 8 * c);
      step[i] = 128;  // 64 bf16 per stage
      dst[i] = WBYTES + xp * 1024;
    }
  }
  auto stage = [&](int j) {
    char* base = smem + (j % NBUF) * SLOT;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
#pragma unroll
      for (int u = 0; u < BKM; ++u) {
        gbl_void_t* from = (gbl_void_t*)(src[i] + (j * BKM + u) * step[i]);
        lds_void_t* to = (lds_void_t*)(base + u * SBYTES + dst[i]);
        if (ONCE && w * LOADS + i < 2 * NF) __builtin_amdgcn_global_load_lds(from, to, 16, 0, 2);   // nt
        else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
      }
  };

  constexpr int SUMS = EPI == SK_F32 ? 4 : 1;
  f32x4 sums[SUMS][FW][TW];
#pragma unroll
  for (int i = 0; i < SUMS; ++i)
#pragma unroll
    for (int f = 0; f < FW; ++f)
#pragma unroll
      for (int t = 0; t < TW; ++t) sums[i][f][t] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int j = 0; j < NBUF - 1; ++j)
    if (j < nst) stage(j);

  auto stream = [&](int j0, int j1) {
    for (int j = j0; j < j1; ++j) {
      // stages j+1 .. min(j+NBUF-2, nst-1) may stay in flight
      wait_stage<LOADS * BKM, NBUF - 2>(min(NBUF - 2, nst - 1 - j));
      if (j + NBUF - 1 < nst) stage(j + NBUF - 1);
#pragma unroll
      for (int u = 0; u < BKM; ++u)
        stage_mma<FW, TW, WBYTES, WROW, EPI == SK_F32>(smem + (j % NBUF) * SLOT + u * SBYTES, sums, wa, wb, lane, g, col);
    }
  };
  if constexpr (EPI == SK_BIAS) {                    // K % (64 BKM slices) == 0
    const int per = nst / sa.slices;
    f32x4 total[FW][TW];
    stream(0, per);
    for (int j0 = per; j0 < nst; j0 += per) {
#pragma unroll
      for (int f = 0; f < FW; ++f)
#pragma unroll
        for (int t = 0; t < TW; ++t) {
          total[f][t] = j0 == per ? sums[0][f][t] : total[f][t] + sums[0][f][t];
          sums[0][f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      stream(j0, j0 + per);
    }
    if (per < nst)
#pragma unroll
      for (int f = 0; f < FW; ++f)
#pragma unroll
        for (int t = 0; t < TW; ++t) sums[0][f][t] = total[f][t] + sums[0][f][t];
  } else {
    stream(0, nst);
  }
  f32x4(&acc)[FW][TW] = sums[0];
  if constexpr (EPI == SK_F32) {
#pragma unroll
    for (int f = 0; f < FW; ++f)
#pragma unroll
      for (int t = 0; t < TW; ++t) acc[f][t] = (acc[f][t] + sums[1][f][t]) + (sums[2][f][t] + sums[3][f][t]);
  }

  if constexpr (SILU) {
    // row group G = n0/16 + wa*FW + f is gate (G even) / up (G odd) of output cols 16*(G/2)..+15
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int m = (wb * TW + t) * 16 + col;
      if (m >= M) continue;
#pragma unroll
      for (int f = 0; f < FW; f += 2) {
        const int G = n0 / 16 + wa * FW + f;
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // same roundings as GEMM -> bf16 gate|up -> silu_mul (HF: silu in the activation dtype)
          const float gt = (float)(bf16)acc[f][t][r], up = (float)(bf16)acc[f + 1][t][r];
          o[r] = (bf16)((float)(bf16)(gt / (1.f + __expf(-gt))) * up);
        }
        *reinterpret_cast<bf16x4*>(Y + (long)m * ldy + (G >> 1) * 16 + 4 * g) = o;
      }
    }
    return;
  }
  if constexpr (EPI == SK_BF16 || EPI == SK_BIAS) {
    // lane holds W rows n = 16f + 4g + r (r = 0..3) for token 16t + col: one 8-B store per fragment
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int m = (wb * TW + t) * 16 + col;
      if (m >= M) continue;
#pragma unroll
      for (int f = 0; f < FW; ++f) {
        const int n = n0 + (wa * FW + f) * 16 + 4 * g;
        if (WROW && n >= N) break;
        bf16x4 o;
        if constexpr (EPI == SK_BIAS) {
          const bf16x4 bv = *reinterpret_cast<const bf16x4*>(sa.bias + n);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bf16 v = (bf16)(acc[f][t][r] + (float)bv[r]);
            o[r] = sa.gelu ? (bf16)gelu_erf((float)v) : v;     // the roundings of gemm_bias_small_kernel
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = (bf16)acc[f][t][r];
        }
        *reinterpret_cast<bf16x4*>(Y + (long)m * ldy + n) = o;
      }
    }
    return;
  }
  if constexpr (EPI == SK_SAMPLE) {
    // token row m's 16*FW columns of this wave sit in lanes col, col+16, col+32, col+48 (g = 0..3):
    // each scores its FW*4, two xor-shuffles inside that lane set (all active or all skipped: they
    // share m), and lane g == 0 leaves the wave's pair
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int m = (wb * TW + t) * 16 + col;
      if (m >= M) continue;
      const float temp = sa.temps[m];
      const bool greedy = !(temp > 0.f);
      const float inv_t = greedy ? 1.f : 1.f / temp;
      const unsigned long long seed = sa.seeds[m];
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int f = 0; f < FW; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int loc = n0 + (wa * FW + f) * 16 + 4 * g + r, idx = sa.voff + loc;
          float v = (float)(bf16)acc[f][t][r];   // the bf16 logit the unfused path samples
          if (!greedy) v = v * inv_t + gumbel_noise(seed, idx);
          if (loc >= sa.vvalid) v = -INFINITY;
          better(bv, bi, v, idx);
        }
#pragma unroll
      for (int o = 16; o < 64; o <<= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        better(bv, bi, ov, oi);
      }
      if (g == 0) {
        const long slot = (long)m * sa.pstride + tile * WA + wa;
        sa.pv[slot] = bv;
        sa.pi[slot] = bi;
      }
    }
    return;
  }
  // lane holds W rows n = 16f + 4g + r (r = 0..3) for token 16t + col: one 16-B store per tile
  float* ps = P + (long)s * Mtot * N + (long)m0 * N;
#pragma unroll
  for (int t = 0; t < TW; ++t) {
    const int m = (wb * TW + t) * 16 + col;
    if (m >= M) continue;
#pragma unroll
    for (int f = 0; f < FW; ++f) {
      const int n = n0 + (wa * FW + f) * 16 + 4 * g;
      if (WROW && n >= N) break;
      *reinterpret_cast<f32x4*>(ps + (long)m * N + n) = acc[f][t];
    }
  }
}

// Y[m, n] = bf16(sum_s P[s, m, n]) (+ R[m, n], rounded like the unfused GEMM-then-add path)
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const float* __restrict__ P, int S, int M, int N,
                                                            bf16* __restrict__ Y, int ldy,
                                                            const bf16* __restrict__ R, int ldr) {
  const long i8 = (long)blockIdx.x * 256 + threadIdx.x;  // index of 8 outputs
  const long total8 = (long)M * N / 8;
  if (i8 >= total8) return;
  const int m = (int)(i8 / (N / 8));
  const int n = (int)(i8 % (N / 8)) * 8;
  float o[8];
  {
    const f32x4* p = reinterpret_cast<const f32x4*>(P + (long)m * N + n);
    const f32x4 a = p[0], b = p[1];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = a[j], o[4 + j] = b[j];
  }
  for (int s = 1; s < S; ++s) {
    const f32x4* p = reinterpret_cast<const f32x4*>(P + ((long)s * M + m) * N + n);
    const f32x4 a = p[0], b = p[1];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] += a[j], o[4 + j] += b[j];
  }
  if (R) {
    float r[8];
    unpack8(*reinterpret_cast<const uint4*>(R + (long)m * ldr + n), r);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (float)(bf16)o[j] + r[j];
  }
  *reinterpret_cast<uint4*>(Y + (long)m * ldy + n) = pack8(o);
}

// wrow bit 0: W is the row-major [N, K] weight (else tile_weight's fragment-tiled copy); bit 1: BK=64
// stages issued in pairs (BKM = 2) -- taken where the ring still holds >= 3 slots and each K slice
// is a multiple of 128, else single stages.  (A double-buffered pair ring -- two slots, for the
// widest tiles at M 97-256 -- measured 3-14 % slower than single stages:
// profiles/r5_decode_gemm_pair_double_buffer_rejected.jsonl.)
template <int NF, int MT, int RKB, int MAXB>
constexpr bool pair_fits() {
  return Ring<NF, MT, RKB, MAXB, 2>::NBUF >= 3;
}

// row-major weights: past the caches in one chunk of rows (ONCE above)
template <int NF, int MT, int WA, int EPI, int MAXB, int BKM, class... A>
void launch_rows(dim3 grid, hipStream_t st, A... args) {
  if constexpr (MT <= 8 && EPI != SK_BIAS) {
    if (grid.y == 1) {
      hipLaunchKernelGGL((splitk_gemm_kernel<NF, MT, WA, EPI, true, 150, MAXB, BKM, true>), grid, dim3(256), 0, st, args...);
      return;
    }
  }
  hipLaunchKernelGGL((splitk_gemm_kernel<NF, MT, WA, EPI, true, 150, MAXB, BKM, false>), grid, dim3(256), 0, st, args...);
}

// one launch of splitk_gemm_kernel<NF, MT, WA, EPI, *, 150, MAXB, *> with the W layout / stage pairing
// of wrow (runtime) mapped onto the template arguments.  ROWS: row-major weights only (the entries whose last tile of columns may be
// part-filled, which the tiled copy's form does not know).
template <int NF, int MT, int WA, int EPI, int MAXB, bool ROWS = false, class... A>
int launch_any(int wrow, bool pair_ok, dim3 grid, hipStream_t st, A... args) {
  const bool rm = wrow & 1;
  if (ROWS && !rm) return (int)hipErrorInvalidValue;
  if constexpr (pair_fits<NF, MT, 150, MAXB>()) {
    if ((wrow & 2) && pair_ok) {
      if (rm) launch_rows<NF, MT, WA, EPI, MAXB, 2>(grid, st, args...);
      else if constexpr (!ROWS) hipLaunchKernelGGL((splitk_gemm_kernel<NF, MT, WA, EPI, false, 150, MAXB, 2>), grid, dim3(256), 0, st, args...);
      return (int)hipGetLastError();
    }
  }
  if (rm) launch_rows<NF, MT, WA, EPI, MAXB, 1>(grid, st, args...);
  else if constexpr (!ROWS) hipLaunchKernelGGL((splitk_gemm_kernel<NF, MT, WA, EPI, false, 150, MAXB>), grid, dim3(256), 0, st, args...);
  return (int)hipGetLastError();
}

template <int NF, int MT, int WA, bool ROWS = false>
int launch(const void* X, int ldx, const void* Wt, int K, float* P, int M, int N, int S, int wrow, hipStream_t st) {
  return launch_any<NF, MT, WA, SK_SLAB, 8, ROWS>(wrow, (K / S) % 128 == 0, dim3(((N + 16 * NF - 1) / (16 * NF)) * S, (M + 16 * MT - 1) / (16 * MT)), st,
                                                  (const bf16*)X, ldx, (const bf16*)Wt, K, P, M, N, S, (bf16*)nullptr, 0, SkSample{});
}

template <int NF, int MT, int WA>
int launch_f32(const void* X, int ldx, const void* W, int K, float* P, int M, int N, int S, int paired, hipStream_t st) {
  const dim3 grid(((N + 16 * NF - 1) / (16 * NF)) * S, (M + 16 * MT - 1) / (16 * MT));
  if constexpr (pair_fits<NF, MT, 150, 16>()) {
    if (paired && (K / S) % 64 == 0) {
      launch_rows<NF, MT, WA, SK_F32, 16, 2>(grid, st, (const bf16*)X, 2 * ldx, (const bf16*)W, 2 * K, P, M, N, S, (bf16*)nullptr, 0, SkSample{});
      return (int)hipGetLastError();
    }
  }
  launch_rows<NF, MT, WA, SK_F32, 16, 1>(grid, st, (const bf16*)X, 2 * ldx, (const bf16*)W, 2 * K, P, M, N, S, (bf16*)nullptr, 0, SkSample{});
  return (int)hipGetLastError();
}

// Y[m, n] = sum_s P[s, m, n], four outputs per thread
__global__ void __launch_bounds__(256) splitk_reduce_f32_kernel(const f32x4* __restrict__ P, int S, long quads, f32x4* __restrict__ Y) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= quads) return;
  f32x4 v = P[i];
  for (int s = 1; s < S; ++s) v += P[s * quads + i];
  Y[i] = v;
}

template <int NF, int MT, int WA>
int launch_silu(const void* X, int ldx, const void* Wt, int K, void* Y, int ldy, int M, int N, int wrow,
                hipStream_t st) {
  return launch_any<NF, MT, WA, SK_SILU, NF == 2 ? 16 : 8>(wrow, K % 128 == 0, dim3(N / (16 * NF), (M + 16 * MT - 1) / (16 * MT)), st, (const bf16*)X,
                                                          ldx, (const bf16*)Wt, K, (float*)nullptr, M, N, 1, (bf16*)Y,
                                                          ldy, SkSample{});
}

template <int NF, int MT, int WA, bool ROWS = false>
int launch_bf16(const void* X, int ldx, const void* Wt, int K, void* Y, int ldy, int M, int N, int wrow,
                hipStream_t st) {
  return launch_any<NF, MT, WA, SK_BF16, 16, ROWS>(wrow, K % 128 == 0, dim3((N + 16 * NF - 1) / (16 * NF), (M + 16 * MT - 1) / (16 * MT)), st,
                                                   (const bf16*)X, ldx, (const bf16*)Wt, K, (float*)nullptr, M, N, 1, (bf16*)Y, ldy, SkSample{});
}

// the streaming LM head: row-major W (wrow) or its fragment-tiled copy; ring budget 150 KiB (one
// workgroup per CU) or 72 KiB (two)
template <int NF, int MT, int WA>
int launch_sample(const void* X, int ldx, const void* Wt, int K, int M, int N, int wrow, int ring2, const SkSample& sa,
                  hipStream_t st) {
  const dim3 grid(N / (16 * NF)), block(256);
#define SK_SAMPLE_LAUNCH(WROW_, KB_)                                                                               \
  hipLaunchKernelGGL((splitk_gemm_kernel<NF, MT, WA, SK_SAMPLE, WROW_, KB_, 16>), grid, block, 0, st, (const bf16*)X, ldx, \
                     (const bf16*)Wt, K, (float*)nullptr, M, N, 1, (bf16*)nullptr, 0, sa)
  // the 72-KiB ring only where it still holds >= 3 stages (else the 150-KiB one)
  constexpr bool R2 = Ring<NF, MT, 72, 16>::NBUF >= 3;
  if constexpr (R2) {
    if (ring2) {
      if (wrow & 1) SK_SAMPLE_LAUNCH(true, 72);
      else SK_SAMPLE_LAUNCH(false, 72);
      return (int)hipGetLastError();
    }
  }
  if (wrow & 1) SK_SAMPLE_LAUNCH(true, 150);
  else SK_SAMPLE_LAUNCH(false, 150);
#undef SK_SAMPLE_LAUNCH
  return (int)hipGetLastError();
}

}  // namespace

// lm_sample_final_kernel's launcher (gemm_prefill.hip): per row, the best of P (score, token) pairs
extern "C" int penny_lm_sample_final(const float* pv, const int* pi, int P, int M, int* out, int* pairs,
                                     hipStream_t stream);

// Fused gate|up + SiLU*up for 16 < M <= 256 (K9 at mid-batch decode): W = tile_weight(interleave16
// gate|up) [N = 2F rows], Y [M, F] bf16 with row stride ldy.  No split-K: N = 28672 already gives
// N/(16*nf) = 224 (nf 8) or 448 (nf 4) workgroups.  M > 256: 256-row token chunks side by side on
// grid y.  Contract (checked): N % (16*nf) == 0, nf in {2, 4, 8}, K % 64 == 0, ldx % 8 == 0, ldy % 4 == 0.
PENNY_API int penny_gateup_silu_gemm(const void* X, int ldx, const void* Wt, int K, void* Y, int ldy, int M, int N,
                                     int nf, int wrow, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > (1 << 20) || K % 64 || ldx % 8 || ldy % 4 || (nf != 2 && nf != 4 && nf != 8) || N % (16 * nf))
    return (int)hipErrorInvalidValue;
  const int mt = min((M + 15) / 16, 16);   // > 256 rows: 256-row token chunks on grid y
  // nf = 2 (one (gate, up) pair per workgroup, WA = 1): twice the workgroups of nf = 4 for narrow
  // TP shards (Llama-3-70B TP=8 gate|up: N = 7168 -> 224 workgroups)
  if (nf == 2) {   // WA = 1 -> 4 token-tile wave columns: token tiles rounded up to a multiple of 4
    if (mt <= 4) return launch_silu<2, 4, 1>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream);
    if (mt <= 8) return launch_silu<2, 8, 1>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream);
    if (mt <= 12) return launch_silu<2, 12, 1>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream);
    return launch_silu<2, 16, 1>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream);
  }
#define GU_CASE(MT_, WA4_, WA8_)                                                          \
  if (mt <= MT_) {                                                                      \
    if (nf == 4) return launch_silu<4, MT_, WA4_>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream); \
    return launch_silu<8, MT_, WA8_>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream);              \
  }
  GU_CASE(2, 2, 2)
  GU_CASE(4, 1, 2)
  GU_CASE(6, 2, 2)
  GU_CASE(8, 1, 2)
  GU_CASE(12, 1, 2)
  GU_CASE(16, 1, 2)
#undef GU_CASE
  return (int)hipErrorInvalidValue;
}

// Shape contract (checked): N % (16*NF) == 0, K % (64*S) == 0, X rows 16-B
// aligned (ldx % 8 == 0).  wrow: bit 0 row-major W instead of tile_weight's copy, bit 1 paired stages.  nf: W row groups per workgroup (2, 4, 6 or 8;
// 6 = 96 rows puts N = 6144 on exactly 64 tiles, i.e. 256 workgroups at S = 4; 16 -- half the X
// bytes per W byte -- measured 5-53 % slower at M = 32-128 on every 8B / TP=8 shape: too few
// workgroups, profiles/r5_decode_gemm_nf16_rejected.jsonl).  P is [S, M, N] f32.
// M > 256: 256-row token chunks side by side on grid y (small prefill steps of narrow TP shards).
PENNY_API int penny_splitk_gemm(const void* X, int ldx, const void* Wt, int K, void* P, int M, int N, int S, int nf,
                                int wrow, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > (1 << 20) || S < 1 || K % (64 * S) || ldx % 8 || (nf != 2 && nf != 4 && nf != 6 && nf != 8) || N % (16 * nf))
    return (int)hipErrorInvalidValue;
  const int mt = min((M + 15) / 16, 16);   // > 256 rows: 256-row token chunks on grid y
  float* p = static_cast<float*>(P);
#define SK_CASE(MT_, WA2_, WA4_, WA8_)                                                 \
  if (mt <= MT_) {                                                                     \
    if (nf == 2) return launch<2, MT_, WA2_>(X, ldx, Wt, K, p, M, N, S, wrow, stream); \
    if (nf == 4) return launch<4, MT_, WA4_>(X, ldx, Wt, K, p, M, N, S, wrow, stream); \
    if (nf == 6) return launch<6, MT_, 2>(X, ldx, Wt, K, p, M, N, S, wrow, stream);    \
    return launch<8, MT_, WA8_>(X, ldx, Wt, K, p, M, N, S, wrow, stream);              \
  }
  // (NF + MT) even; wave split picked to minimise fragment reads per wave (NF/WA + MT/WB)
  SK_CASE(2, 2, 2, 2)
  SK_CASE(4, 1, 1, 2)
  SK_CASE(6, 2, 2, 2)
  SK_CASE(8, 1, 1, 2)
  SK_CASE(12, 1, 1, 2)
  SK_CASE(16, 1, 1, 2)
#undef SK_CASE
  return (int)hipErrorInvalidValue;
}

// Split-K gate|up: P [S, M, N] f32 slabs of the interleave16 gate|up projection (row group 2j = gate
// features 16j..16j+15, 2j+1 = their up rows) -> Y [M, N/2] bf16 = silu(gate) * up with the SK_SILU
// epilogue's roundings.  For gate|up shapes whose column tiles alone underfill the chip (Llama-3-70B
// TP=8 shard: 7168 rows = 112 tiles at nf = 4) or whose weights stream row-major (70B TP=1: no tiled
// copy), the K split fills the CUs and this pass adds S*8 B per output.  One thread per 8 outputs.
__global__ void __launch_bounds__(256) splitk_reduce_silu_kernel(const float* __restrict__ P, int S, int M, int N,
                                                                 bf16* __restrict__ Y, int ldy) {
  const int F = N / 2;
  const long i8 = (long)blockIdx.x * 256 + threadIdx.x;  // index of 8 outputs
  const long total8 = (long)M * F / 8;
  if (i8 >= total8) return;
  const int m = (int)(i8 / (F / 8));
  const int f = (int)(i8 % (F / 8)) * 8;                 // 8 features of one 16-feature group
  const int ng = (f >> 4) * 32 + (f & 15);               // gate column; up = ng + 16
  float gt[8], up[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) gt[j] = up[j] = 0.f;
  for (int s = 0; s < S; ++s) {
    const f32x4* pg = reinterpret_cast<const f32x4*>(P + ((long)s * M + m) * N + ng);
    const f32x4* pu = reinterpret_cast<const f32x4*>(P + ((long)s * M + m) * N + ng + 16);
    const f32x4 g0 = pg[0], g1 = pg[1], u0 = pu[0], u1 = pu[1];
#pragma unroll
    for (int j = 0; j < 4; ++j) gt[j] += g0[j], gt[4 + j] += g1[j], up[j] += u0[j], up[4 + j] += u1[j];
  }
  float o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float gb = (float)(bf16)gt[j], ub = (float)(bf16)up[j];
    o[j] = (float)(bf16)(gb / (1.f + __expf(-gb))) * ub;
  }
  *reinterpret_cast<uint4*>(Y + (long)m * ldy + f) = pack8(o);
}

PENNY_API int penny_splitk_reduce_silu(const void* P, int S, int M, int N, void* Y, int ldy, hipStream_t stream) {
  if (M <= 0) return 0;
  if (N % 32 || ldy % 8 || S < 1) return (int)hipErrorInvalidValue;
  const long total8 = (long)M * (N / 2) / 8;
  hipLaunchKernelGGL(splitk_reduce_silu_kernel, dim3((unsigned)((total8 + 255) / 256)), dim3(256), 0, stream,
                     (const float*)P, S, M, N, (bf16*)Y, ldy);
  return (int)hipGetLastError();
}

PENNY_API int penny_splitk_reduce(const void* P, int S, int M, int N, void* Y, int ldy, const void* R, int ldr,
                                  hipStream_t stream) {
  if (M <= 0) return 0;
  if (N % 8 || ldy % 8 || (R && ldr % 8)) return (int)hipErrorInvalidValue;
  const long total8 = (long)M * N / 8;
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((total8 + 255) / 256)), dim3(256), 0, stream,
                     (const float*)P, S, M, N, (bf16*)Y, ldy, (const bf16*)R, ldr);
  return (int)hipGetLastError();
}

// Row-parallel decode projection with a bf16 output (no split-K): Y [M, N] (row stride ldy) =
// X [M, K] x W [N, K]^T, one workgroup per 16*nf W rows -- the TP shards of O / down whose output
// feeds the all-reduce directly (Llama-3-70B TP=8: N = 8192 -> 256 workgroups at nf = 2).
// Contract (checked): N % (16*nf) == 0, nf in {2, 4, 8}, K % 64 == 0, ldx % 8 == 0, ldy % 4 == 0,
// M >= 1 (> 256: 256-row token chunks on grid y).
PENNY_API int penny_splitk_gemm_bf16(const void* X, int ldx, const void* Wt, int K, void* Y, int ldy, int M, int N,
                                     int nf, int wrow, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > (1 << 20) || K % 64 || ldx % 8 || ldy % 4 || (nf != 2 && nf != 4 && nf != 8) || N % (16 * nf))
    return (int)hipErrorInvalidValue;
  const int mt = min((M + 15) / 16, 16);   // > 256 rows: 256-row token chunks on grid y
#define BF_CASE(MT_, WA2_, WA4_, WA8_)                                                          \
  if (mt <= MT_) {                                                                            \
    if (nf == 2) return launch_bf16<2, MT_, WA2_>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream);  \
    if (nf == 4) return launch_bf16<4, MT_, WA4_>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream);  \
    return launch_bf16<8, MT_, WA8_>(X, ldx, Wt, K, Y, ldy, M, N, wrow, stream);               \
  }
  BF_CASE(2, 2, 2, 2)
  BF_CASE(4, 1, 1, 2)
  BF_CASE(6, 2, 2, 2)
  BF_CASE(8, 1, 1, 2)
  BF_CASE(12, 1, 1, 2)
  BF_CASE(16, 1, 1, 2)
#undef BF_CASE
  return (int)hipErrorInvalidValue;
}

namespace {

// What a block of penny_linear_rows takes for 2048 of K beyond its fixed 2.8 us, by its 16 nf columns and 16 mt rows
struct RowsTile {
  int nf, mt;
  float us, us32;                        // bf16, f32 (the tiles that f32 takes)
};
constexpr RowsTile kRowsTiles[] = {{2, 2, 4.6f, 13.6f}, {2, 4, 6.5f, 23.4f}, {4, 2, 6.7f, 24.4f}, {2, 6, 8.2f, 33.f}, {4, 4, 9.8f, 0.f},
                                   {2, 8, 9.9f, 0.f},   {4, 6, 11.7f, 0.f},  {8, 2, 12.3f, 0.f},  {4, 8, 15.f, 0.f},  {8, 4, 15.3f, 0.f},
                                   {8, 6, 21.f, 0.f},   {4, 12, 19.2f, 0.f}, {8, 8, 24.f, 0.f}};

}  // namespace

// The tile and split of penny_linear_rows for M rows: nf | mt << 8 | S << 16, or 0 where another product is to be taken (best: its time).
//
// A block's ring takes a CU's LDS, so the blocks run in rounds of 256, each round for as long as its tile's K: a product is the
// faster the smaller the tile, as long as one round holds all blocks; with few blocks K is cut in 2 or 4 (a second launch and
// a pass over the slabs: 2 us and 1 us per MB).  Against the library, weights beyond the caches, us library / here: 2048 x 4096
// 1 row 14.8 / 8.4, 64 13.9 / 10.1; 4096 x 2048 64 12.2 / 8.7, 256 13.7 / 13.7; 7232 x 2048 64 12.9 / 11.4, 256 24.2 / 19.9; 12864 x 2048 64 16.1 /
// 15.4, 160 24.6 / 23.6; 2048 x 2048 64 8.9 / 7.2, 256 9.9 / 9.8, 512 12.0 / 13.0; 6464 x 1024 64 11.7 / 7.3, 256 15.1 / 12.0; 2048 x 1024 256 8.7 / 6.4, 768
// 10.1 / 9.4; 1024 x 3072 64 10.0 / 7.0, 256 9.1 / 10.3; 1024 x 1024 64 8.6 / 5.1, 512 8.6 / 6.4.  A library call costs the host 20 - 24 us as well,
// this one 8: a step of many small launches is bounded by that.  So products of up to 20 us are taken up to 512 rows, where some
// are up to a tenth slower than the library's, and from there, as the device becomes the bound, ever shorter ones, to 16 us at 1024
// rows and 8 at 2048.  Whole passes of 400, 600 and 1000 tokens, three hybrid decoders of width 1024, us: 1538 -> 1086, 1739 -> 1347, 1399 ->
// 935; 1540 -> 1160, 1730 -> 1378, 1440 -> 976; 1570 -> 1399, 1790 -> 1526, 1505 -> 1125; width 2048 at 400: 1811 -> 1789, 1789 -> 1769, 1657
// -> 1650.  Up to 96 rows, the steps of captured decodes, all but the longest are taken (14912 x 2048, 96 rows: 18.7 / 18.3).
//
// f32 (a sixteenth of the matrix rate; the four smallest tiles): the library's tiles are 1.1 - 1.3 times faster from 40 - 100 rows on where
// the device counts (1024 x 3072, 64 rows 10.6 / 12.3; 2048 x 1024 at 150 11.4 / 14.7) and slower below (1024 x 1024 1 row 8.3 / 6.2, 64 8.7 / 7.3;
// 2048 x 1024 16 rows 8.8 / 6.9; 1024 x 3072 10.9 / 9.0), so up to 64 rows, which may be a captured step, the products of up to 11 us are taken, and
// beyond, where the host is the bound, up to 20.  Steps at width 1024: 14 rows decoding 956 -> 812, 50 1023 -> 916; prompts (11 us up to 256 rows / 20):
// 74 tokens 1472 / 1141, 150 beside 9 rows 1457 / 1177, 120 beside 4 1423 / 1220, 100 beside 6 1277 / 1114, 200 1440 / 1349 (of which the widths of
// 3112 - 4136 that are no multiples of 16 a part; decoding in bf16 they alone are 30 rows 677 / 625 and 695 / 649).  Errors against 64 bits at most the library's
// (K = 1024 1.6 - 2.9e-7 of the norm against 2.9 - 5.8e-7, K = 3072 2.0 - 2.6e-7 against 5.0e-7).
//
// Beyond 256 rows of f32 the device's time meets the host's, and the line falls with the rows as that of bf16 does: from 20 us to 14.7 at 384, from
// where whole passes are level or behind (none beyond 256 rows / this line; 8 layers of width 1024, two hybrid decoders and one whose passes the device bounds
// earlier): 270 rows 1620 / 1480, 1604 / 1411, 1608 / 1505; 320 1624 / 1490, 1710 / 1531, 1628 / 1653; 350 1624 / 1600, 1696 / 1520, 1656 / 1674; 384 1631 /
// 1642, 1689 / 1524, 1722 / 1743; products of up to 15 us at 400 rows 1778 / 1807, 1682 / 1630, 1762 / 1776, at 512 1784 / 1811, 1682 / 1717, 1901 / 1919.
static int rows_plan(int M, int N, int K, int f32, float& best) {
  if (M <= 0 || M > (f32 ? 384 : 2048) || N < 512 || N % 8 || K <= 0 || K % (f32 ? 32 : 64)) return 0;
  int plan = 0;
  best = f32 ? (M <= 64 ? 11.f : M <= 256 ? 20.f : 20.f - (M - 256) / 24.f) : M <= 96 ? 60.f : M <= 512 ? 20.f : 20.f - (M - 512) / 128.f;
  for (int S = 1; S <= (f32 ? 8 : 4); S *= 2) {
    if (S > 1 && (K % (64 * S) || K / S < 256)) break;
    for (int i = 0; i < (f32 ? 4 : (int)(sizeof(kRowsTiles) / sizeof(kRowsTiles[0]))); ++i) {
      const RowsTile& t = kRowsTiles[i];
      const long blocks = (long)((N + 16 * t.nf - 1) / (16 * t.nf)) * ((M + 16 * t.mt - 1) / (16 * t.mt)) * S;
      if (S > 1 && blocks > 256) continue;
      const float us = (blocks + 255) / 256 * (2.8f + (f32 ? t.us32 : t.us) * (K / S) / 2048.f) + (S > 1 ? 2.f + 4e-6f * S * M * N : 0.f);
      if (us < best) best = us, plan = t.nf | t.mt << 8 | S << 16;
    }
  }
  return plan;
}

PENNY_API int penny_linear_rows_plan(int M, int N, int K, int f32) {
  float us;
  return f32 && M > 256 ? 0 : rows_plan(M, N, K, f32, us);
}
// f32 of any number of rows: the rows beyond 256 are for calls whose host's time counts, no launches that a graph replays
PENNY_API int penny_linear_rows_f32_plan(int M, int N, int K) {
  float us;
  return rows_plan(M, N, K, 1, us);
}
// the estimate of the plan for bf16, FLT_MAX where there is none
extern "C" float penny_linear_rows_us(int M, int N, int K) {
  float us;
  return rows_plan(M, N, K, 0, us) ? us : FLT_MAX;
}

// The same for launches that a graph replays, where the host's share of a library call does not count: only what the device runs faster.
// Up to 96 rows (f32: 32) that is all of the above.  Beyond, us in replayed graphs, library / here: bf16 7232 x 2048 160 rows 17.4 / 16.1, 256
// 24.8 / 20.2; 4096 x 2048 192 21.5 / 12.4; 6464 x 1024 256 15.0 / 12.0; 2048 x 6144 (in slices) 192 22.6 / 17.7; but 2048 x 4096 unsplit 192 15.9 / 16.7, 12864
// x 2048 128 19.5 / 21.2, 32000 x 1024 128 18.8 / 20.5.  f32 2048 x 1024 48 11.3 / 9.9, 1024 x 2048 64 11.3 / 10.6, 2048 x 32 256 3.9 / 3.1; but 1024 x 3072 48
// 10.9 / 12.4, 3616 x 1024 48 12.1 / 12.6, 1024 x 1024 80 8.2 / 9.0, 256 8.8 / 11.2, 2048 x 1024 128 11.6 / 11.8.
PENNY_API int penny_linear_rows_replay_plan(int M, int N, int K, int f32) {
  const int plan = penny_linear_rows_plan(M, N, K, f32);
  if (M <= (f32 ? 32 : 96)) return plan;
  if (f32) return K <= 64 || (M <= 64 && (long)N * K <= 2048 * 1024) ? plan : 0;
  return N <= 8192 && (K < 4096 || plan >> 16 > 1) ? plan : 0;
}

#define ROWS_TILES(CASE) \
  CASE(2, 2, 2) CASE(2, 4, 1) CASE(4, 2, 2) CASE(2, 6, 2) CASE(4, 4, 1) CASE(2, 8, 1) CASE(4, 6, 2) CASE(8, 2, 2) CASE(4, 8, 1) CASE(8, 4, 2) \
  CASE(8, 6, 2) CASE(4, 12, 1) CASE(8, 8, 2)

// S slices of K of X W^T (bf16, W row-major) to f32 slabs [S, M, N]
extern "C" int penny_rows_slabs(const void* X, int ldx, const void* W, int K, float* slabs, int M, int N, int S, int nf, int mt, int paired,
                                hipStream_t st) {
  if (M <= 0) return 0;
  if (M > (1 << 20) || N <= 0 || N % 8 || S < 1 || K <= 0 || K % (64 * S) || ldx % 8) return (int)hipErrorInvalidValue;
#define SLABS_CASE(NF_, MT_, WA_) \
  if (nf == NF_ && mt == MT_) return launch<NF_, MT_, WA_, true>(X, ldx, W, K, slabs, M, N, S, paired ? 3 : 1, st);
  ROWS_TILES(SLABS_CASE)
#undef SLABS_CASE
  return (int)hipErrorInvalidValue;
}

// Y [M, N] = X [M, K] x W [N, K]^T in bf16 or f32 (f32 != 0) for up to about two thousand rows, W row-major: slabs == null streams W once (S = 1), else
// S slices of K leave f32 slabs [S, M, N] that a second launch adds, or with Y null the reader.  One entry for both, so that a step that
// the host bounds pays for one call.  nf, mt: a block's columns and rows in units of 16, one of kRowsTiles.  Contract (checked): N % 8 == 0 (the last
// tile may be part-filled), K % (64 * S) == 0 (f32: 32 * S), rows of x in whole 16 bytes, y contiguous.
PENNY_API int penny_linear_rows(const void* X, int ldx, const void* W, int K, void* Y, int M, int N, void* slabs, int S, int nf, int mt,
                                int f32, int paired, hipStream_t st) {
  if (M <= 0) return 0;
  if (M > (1 << 20) || N <= 0 || N % 8 || S < 1 || (S > 1) != (slabs != nullptr) || (S == 1 && Y == nullptr) || K <= 0 ||
      K % ((f32 ? 32 : 64) * S) || K > (1 << 28) || ldx % (f32 ? 4 : 8))
    return (int)hipErrorInvalidValue;
  float* p = static_cast<float*>(f32 && S == 1 ? Y : slabs);
  int rc;
#define LR_CASE(NF_, MT_, WA_)                                                                     \
  if (nf == NF_ && mt == MT_) {                                                                    \
    if (f32) {                                                                                     \
      if constexpr (NF_ * MT_ <= 12) rc = launch_f32<NF_, MT_, WA_>(X, ldx, W, K, p, M, N, S, paired, st); \
      else return (int)hipErrorInvalidValue;                                                       \
    } else if (S > 1) {                                                                            \
      rc = penny_rows_slabs(X, ldx, W, K, p, M, N, S, nf, mt, paired, st);                         \
    } else {                                                                                       \
      rc = launch_bf16<NF_, MT_, WA_, true>(X, ldx, W, K, Y, N, M, N, paired ? 3 : 1, st);         \
    }                                                                                              \
  } else
  ROWS_TILES(LR_CASE)
  return (int)hipErrorInvalidValue;
#undef LR_CASE
  if (rc || S == 1 || Y == nullptr) return rc;
  if (!f32) return penny_splitk_reduce(slabs, S, M, N, Y, N, nullptr, 0, st);
  const long quads = (long)M * N / 4;
  splitk_reduce_f32_kernel<<<dim3((unsigned)((quads + 255) / 256)), 256, 0, st>>>((const f32x4*)slabs, S, quads, (f32x4*)Y);
  return (int)hipGetLastError();
}

// The tile of penny_bias_rows (S = 1) or penny_rows_slabs for M rows: the fastest that runs all its blocks in one round; 0: none does
extern "C" int penny_bias_rows_tile(int M, int N, int S) {
  int tile = 0;
  float best = 1e9f;
  for (const RowsTile& t : kRowsTiles) {
    const long blocks = (long)((N + 16 * t.nf - 1) / (16 * t.nf)) * ((M + 16 * t.mt - 1) / (16 * t.mt)) * S;
    if (blocks <= 256 && t.us < best) best = t.us, tile = t.nf | t.mt << 8;
  }
  return tile;
}

// ... and what it takes, by the figures above
extern "C" float penny_bias_rows_us(int M, int N, int K) {
  const int tile = penny_bias_rows_tile(M, N, 1);
  for (const RowsTile& t : kRowsTiles)
    if (tile == (t.nf | t.mt << 8)) return 2.8f + t.us * K / 2048.f;
  return FLT_MAX;
}

// Y [M, N] (row stride ldy) = bf16(X W^T + bias) [-> exact GELU] on the same tiles, for penny_gemm_bias_small; the sums are those of
// penny_rows_slabs in `slices` slices, added in turn
extern "C" int penny_bias_rows(const void* X, int ldx, const void* W, int K, void* Y, int ldy, const void* bias, int M, int N, int gelu, int slices, int nf,
                               int mt, hipStream_t st) {
  if (M <= 0) return 0;
  if (M > (1 << 20) || N <= 0 || N % 16 || K <= 0 || slices < 1 || K % (64 * slices) || ldx % 8 || ldy % 4)
    return (int)hipErrorInvalidValue;
  SkSample sa{};
  sa.bias = static_cast<const bf16*>(bias);
  sa.gelu = gelu;
  sa.slices = slices;
#define BR_CASE(NF_, MT_, WA_)                                                                                          \
  if (nf == NF_ && mt == MT_)                                                                                           \
    return launch_any<NF_, MT_, WA_, SK_BIAS, 16, true>(3, K / slices % 128 == 0, dim3((N + 16 * NF_ - 1) / (16 * NF_), (M + 16 * MT_ - 1) / (16 * MT_)), \
                                                  st, (const bf16*)X, ldx, (const bf16*)W, K, (float*)nullptr, M, N, 1, (bf16*)Y, ldy, sa);
  ROWS_TILES(BR_CASE)
#undef BR_CASE
  return (int)hipErrorInvalidValue;
}

// Weight-streaming LM head + sampler (K11 + K12) for decode batches, full vocabulary or a TP rank's
// padded shard: W [Vpad, K] (row-major with wrow = 1, else tile_weight's copy) holds global rows
// voff .. voff + vvalid - 1 then padding; per row m the Gumbel-max (temps[m] > 0) / argmax sample.
// out [M] int32 (the token) and/or pairs [M, 2] int32 (score bits, global id: the shard's candidate).
// workspace >= 2 * M * (Vpad / (16*nf)) * 2 floats.  ring2: the 72-KiB ring (two workgroups per CU).
// Contract (checked): 1 <= M <= 128, Vpad % (16*nf) == 0, nf in {4, 8}, 0 < vvalid <= Vpad,
// K % 64 == 0, ldx % 8 == 0.
PENNY_API int penny_lm_head_stream_sample(const void* X, int ldx, const void* W, int K, int M, int Vpad, int vvalid,
                                          int voff, const float* temps, const unsigned long long* seeds,
                                          void* workspace, int* out, int* pairs, int nf, int wrow, int ring2,
                                          hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 128 || (nf != 4 && nf != 8) || Vpad % (16 * nf) || vvalid <= 0 || vvalid > Vpad || voff < 0 || K % 64 ||
      ldx % 8 || !temps || !seeds || !workspace || (!out && !pairs))
    return (int)hipErrorInvalidValue;
  const int tiles = Vpad / (16 * nf), mt = (M + 15) / 16;
  // wave split per (nf, token tiles): as penny_splitk_gemm's table
  const int wa = nf == 8 ? 2 : (mt <= 2 || (mt > 4 && mt <= 6) ? 2 : 1);
  const int pstride = tiles * wa;
  float* pv = static_cast<float*>(workspace);
  int* pi = reinterpret_cast<int*>(pv + (long)M * pstride);
  const SkSample sa{temps, seeds, pv, pi, pstride, voff, vvalid};
  int rc;
#define LS_CASE(MT_, WA4_)                                                                                      \
  if (mt <= MT_) {                                                                                              \
    if (nf == 4) rc = launch_sample<4, MT_, WA4_>(X, ldx, W, K, M, Vpad, wrow, ring2, sa, stream);              \
    else rc = launch_sample<8, MT_, 2>(X, ldx, W, K, M, Vpad, wrow, ring2, sa, stream);                          \
  } else
  LS_CASE(2, 2)
  LS_CASE(4, 1)
  LS_CASE(6, 2)
  LS_CASE(8, 1)
  return (int)hipErrorInvalidValue;
#undef LS_CASE
  if (rc) return rc;
  return penny_lm_sample_final(pv, pi, pstride, M, out, pairs, stream);
}
