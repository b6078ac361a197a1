// Routed feed-forwards: the chosen experts of every token as two grouped matrix products over rows sorted by expert,
//     act[r] = unit(W1[e] x[token(r)])      W1 [N1, W] per expert (gated: gate and up rows in turns of 16)
//     ys[r]  = W2[e] act[r]                 W2 [W, F] per expert
// At most three launches and no host read of the bucket sizes:
//   plan    a stable counting sort of the (token, choice) pairs by expert and the list of row tiles: one block, beyond 1024 pairs one
//           per expert; no launch of its own for up to 1024 pairs in the stream form below
//   GEMM 1  gathers the tokens' rows while it stages them, applies the gated unit in its epilogue
//   GEMM 2  sorted rows in and out; mx_moe_combine sums a token's rows
// Weights are stored as the MFMA reads them: pieces of 1 KiB, [row group of 16][K step of 64 bytes][64 lanes][16 B],
// lane l holding row l % 16 and the 16 bytes at 16 * (l / 16); rows and K padded with zeros (whole groups, K to 128 B).
// Both storage types share the code: a 16-byte operand is 8 bf16 (one 16x16x32 MFMA) or 4 f32 (four 16x16x4 MFMAs whose
// step j takes K element 4 g + j of both operands).  Accumulation is f32; the unit sees the f32 sums.
//
// Three forms, chosen by the rows an expert gets on average (the bucket sizes stay on the device):
//   tile    128 W rows x 64, 128 or 192 tokens per block (64 x 64 for few in f32), both operands through an LDS ring of two or three stages
//           filled by LDS-DMA, two or three blocks per CU: bound by the operand reads.  4096 tokens, width 2048, 32 experts of 1024, top 4,
//           bf16: 300 us for both products (650 TFLOP/s); 31 pairs of library products and the host's wait for the
//           bucket sizes took 1.3 ms.
//   wide    256 W rows x 256 tokens per block, bf16: bound by the matrix cores and, with few rounds of blocks, by the last one
//           (5065 tokens of the same layer: 366 -> 315 us, 8192: 515 -> 420, 930 TFLOP/s).
//   stream  32 or 64 W rows x 16 tokens per block, the four waves split K and the weights go straight to registers,
//           1 KiB per load: bound by the weight stream.  64 tokens of the same layer: 49 + 23 us, 5.5 and 5.9 TB/s
//           (batched library products of all rows with all experts, their unit and combine: 125 us).
#include <math.h>

#include "mx_common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int N> struct Steps { static constexpr int value = N; };

enum { UNIT_NONE = 0, UNIT_CLAMP = 1, UNIT_SILU = 2, UNIT_GELU = 3, UNIT_RELU2 = 4 };

// 16 zero bytes: what a lane stages for K positions behind a row's end
__device__ uint4 g_zero16;

struct ExpertGemm {
  const void* x;        // rows of ldx elements: token rows (top > 0: sorted row r reads row src[r] / top) or sorted rows
  long ldx;
  int kbytes;           // bytes of a row that count
  const int* src;       // sorted row -> pair
  int top;
  const int4* tiles;    // (expert, first sorted row, rows, -), then entries without rows; the one before the first: how many have
                        // rows, how many of them more than half a tile of 256
  int ntiles;           // entries of the list
  const char* w;        // pieces, expert stride wstride bytes
  long wstride;
  int kt;               // pieces per row group
  int groups;           // row groups
  void* y;              // sorted rows of ldy elements, columns 0 .. ncol - 1 written
  long ldy;
  int ncol;
  int unit;
  float limit, alpha;
  const float* scale;   // per pair, on the expert's input (or null)
  // stream form with a plan of its own (plan_tile): the pairs' experts (null: without), and where the plan goes for what comes after
  const int* idx;
  int pairs, experts;
  int *pos, *src_out;
  int4* tiles_out;
};

// Rows of each of the tiles of an expert with c rows but the last, which has the rest: even shares in whole groups of 16, as the tile form's
// blocks cost what they hold and the longest is waited for (5065 tokens in tiles of 192 351 -> 337 us, 3453 254 -> 249; tiles of 128
// level); tiles of 256 cost halves
__device__ __forceinline__ int tile_share(int c, int mt) {
  const int k = max((c + mt - 1) / mt, 1);
  return mt == 256 ? mt : ((c + k - 1) / k + 15) / 16 * 16;
}

// One block: pairs 0 .. P-1 (expert idx[i], identity experts >= E stay out) in a stable order by expert.  Every wave
// owns a contiguous run of pairs; lanes with equal experts find each other by ballots over the index bits, so no
// atomics, and pos / src are the same on every run.  Bound by latency: NC > 0 keeps a wave's run of NC * 64 indices in
// registers, all loads in flight at once (16,384 pairs: 34 us as a loop over memory).  LDS: cnt [waves][E], base [E].
template <int NC>
__global__ void __launch_bounds__(1024) expert_plan_kernel(const int* __restrict__ idx, int P, int E, int bits, int mt,
                                                           int ntiles, int* __restrict__ pos, int* __restrict__ src,
                                                           int4* __restrict__ tiles) {
  extern __shared__ int lds[];
  const int nw = blockDim.x >> 6, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int* cnt = lds + w * E;
  int* base = lds + nw * E;
  const int per = NC > 0 ? NC * 64 : (P + nw * 64 - 1) / (nw * 64) * 64, i0 = w * per, i1 = min(P, i0 + per);
  const int nc = NC > 0 ? NC : (i1 - i0 + 63) / 64;
  int held[NC > 0 ? NC : 1];
#pragma unroll
  for (int c = 0; c < NC; ++c) held[c] = i0 + c * 64 + lane < i1 ? idx[i0 + c * 64 + lane] : E;
  auto expert = [&](int c) { return NC > 0 ? held[c] : (i0 + c * 64 + lane < i1 ? idx[i0 + c * 64 + lane] : E); };
  for (int e = threadIdx.x; e < nw * E; e += blockDim.x) lds[e] = 0;
  __syncthreads();
  auto peers = [&](int e) {
    unsigned long long m = __ballot(e < E);
    for (int b = 0; b < bits; ++b) {
      const unsigned long long s = __ballot((e >> b) & 1);
      m &= (e >> b) & 1 ? s : ~s;
    }
    return m;
  };
#pragma unroll
  for (int c = 0; c < nc; ++c) {
    const int e = expert(c);
    const unsigned long long m = peers(e);
    if (e < E && __ffsll(m) - 1 == lane) cnt[e] += __popcll(m);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) {        // this expert's first place per wave, and its total
    int t = 0;
    for (int v = 0; v < nw; ++v) {
      const int c = lds[v * E + e];
      lds[v * E + e] = t;
      t += c;
    }
    base[e] = t;
  }
  __syncthreads();
  if (w == 0) {                                              // exclusive sums over the experts: rows and tiles
    int rows = 0, nt = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane, c = e < E ? base[e] : 0, t = (c + mt - 1) / mt;
      int sc = c, st = t;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int a = __shfl_up(sc, o, 64), b = __shfl_up(st, o, 64);
        if (lane >= o) sc += a, st += b;
      }
      const int r0 = rows + sc - c, t0 = nt + st - t;
      if (e < E) base[e] = r0;
      const int share = tile_share(c, mt);
      for (int k = 0; k < t; ++k)
        if (t0 + k < ntiles) tiles[t0 + k] = make_int4(e, r0 + k * share, min(share, c - k * share), 0);
      rows += __shfl(sc, 63, 64);
      nt += __shfl(st, 63, 64);
    }
    for (int t = nt + lane; t < ntiles; t += 64) tiles[t] = make_int4(0, 0, 0, 0);
    if (lane == 0) tiles[-1] = make_int4(nt, nt, 0, 0);
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < nc; ++c) {
    const int i = i0 + c * 64 + lane, e = expert(c);
    const unsigned long long m = peers(e);
    if (e < E) {
      const int at = base[e] + cnt[e] + __popcll(m & ((1ull << lane) - 1));
      pos[i] = at;
      src[at] = i;
    } else if (i < i1) {
      pos[i] = 0;
    }
    __builtin_amdgcn_wave_barrier();                         // every lane has read its count
    if (e < E && __ffsll(m) - 1 == lane) cnt[e] += __popcll(m);
    __builtin_amdgcn_wave_barrier();
  }
}

// The same plan by one block per expert, for more pairs than one block sorts in the time of a launch.  Every block counts all
// pairs (LDS atomics into a row of bins per wave), so it knows its expert's first row and tile without the other blocks, and
// then places its own expert's pairs: one ballot per chunk of 64 instead of one per bit of the index.  Same pos and src as
// above, and the same tiles, but that tiles of 256 rows at most half full come last.  Bound by the latency of reading the indices
// and of the count.  Us in one block / here, 32 experts: 20,260 pairs 30.7 / 9.6, 4,736: 10.5 / 4.9, 2,048: 4.6 / 4.1, 1,536: 4.5 /
// 4.0, 1,024 and fewer: alike; 8 and 256 experts draw the same line (1,024 pairs 3.8 / 3.8 and 6.6 / 6.6, 4,096: 7.6 / 4.7 and 13.8 /
// 4.8).  NC > 0: NC * 1024 pairs at most, held in registers; 0: any number, read twice.  LDS: cnt [16][E], total [E].
template <int NC>
__global__ void __launch_bounds__(1024) expert_plan_wide_kernel(const int* __restrict__ idx, int P, int E, int mt, int ntiles,
                                                                int* __restrict__ pos, int* __restrict__ src,
                                                                int4* __restrict__ tiles) {
  extern __shared__ int lds[];
  __shared__ int own[4];                                     // first row, first tile, first tile of the last ones, full tiles
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, me = blockIdx.x;
  int* cnt = lds + w * E;
  int* total = lds + 16 * E;
  const int nc = NC > 0 ? NC : (P + 1023) / 1024, i0 = w * nc * 64 + lane;
  int held[NC > 0 ? NC : 1];
#pragma unroll
  for (int c = 0; c < NC; ++c) held[c] = i0 + c * 64 < P ? idx[i0 + c * 64] : -1;
  auto expert = [&](int c) { return NC > 0 ? held[c] : (i0 + c * 64 < P ? idx[i0 + c * 64] : -1); };
  for (int e = threadIdx.x; e < 16 * E; e += 1024) lds[e] = 0;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < nc; ++c) {
    const int e = expert(c);
    if ((unsigned)e < (unsigned)E) atomicAdd(cnt + e, 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 1024) {
    int t = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v) t += lds[v * E + e];
    total[e] = t;
  }
  __syncthreads();
  const int half = mt == 256 ? 128 : 0;
  auto begun = [&](int c) { return c % mt != 0 && c % mt <= half; };       // the last tile is one of the small ones
  if (w == 0) {
    int rows = 0, full = 0, small = 0, fulls = 0, smalls = 0;
    for (int e = lane; e < E; e += 64) {
      const int c = total[e], sm = begun(c), fl = (c + mt - 1) / mt - sm;
      if (e < me) rows += c, full += fl, small += sm;
      fulls += fl;
      smalls += sm;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      rows += __shfl_xor(rows, o, 64), full += __shfl_xor(full, o, 64), small += __shfl_xor(small, o, 64);
      fulls += __shfl_xor(fulls, o, 64), smalls += __shfl_xor(smalls, o, 64);
    }
    if (lane == 0) {
      own[0] = rows, own[1] = full, own[2] = fulls + small, own[3] = fulls + smalls;
      if (me == 0) tiles[-1] = make_int4(fulls + smalls, fulls, 0, 0);
    }
  }
  __syncthreads();
  const int row0 = own[0], tile0 = own[1], small0 = own[2], all = own[3], n = total[me];
  const int share = tile_share(n, mt);
  for (int k = threadIdx.x; k * mt < n; k += 1024) {
    const int at = n - k * mt < mt && begun(n) ? small0 : tile0 + k;
    if (at < ntiles) tiles[at] = make_int4(me, row0 + k * share, min(share, n - k * share), 0);
  }
  if (me == 0)
    for (int t = all + threadIdx.x; t < ntiles; t += 1024) tiles[t] = make_int4(0, 0, 0, 0);
  int at = row0;
  for (int v = 0; v < w; ++v) at += lds[v * E + me];
#pragma unroll
  for (int c = 0; c < nc; ++c) {
    const int e = expert(c);
    const unsigned long long m = __ballot(e == me);
    if (e == me) {
      const int r = at + __popcll(m & ((1ull << lane) - 1));
      pos[i0 + c * 64] = r;
      src[r] = i0 + c * 64;
    } else if (me == 0 && e >= E) {
      pos[i0 + c * 64] = 0;
    }
    at += __popcll(m);
  }
}

__device__ __forceinline__ float unit_value(int unit, float g, float u, float limit, float alpha) {
  if (unit == UNIT_CLAMP) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g * mx_sigmoid(alpha * g) * (u + 1.0f);
  }
  if (unit == UNIT_SILU) return mx_silu(g) * u;
  const float z = 0.7978845608028654f * (g + 0.044715f * g * g * g);   // gelu, tanh form
  return 0.5f * g * (1.0f + mx_tanh(z)) * u;
}

// four adjacent output columns c .. c + 3 of sorted row r: gate and up sums, or one sum
template <typename T, bool GLU>
__device__ __forceinline__ void expert_store(const ExpertGemm& a, long r, int c, f32x4 g, f32x4 u, int pair = -1) {
  if (c >= a.ncol) return;
  typedef T vec __attribute__((ext_vector_type(4)));
  if (GLU && a.scale != nullptr) {
    const float s = a.scale[pair >= 0 ? pair : a.src[r]];
#pragma unroll
    for (int j = 0; j < 4; ++j) g[j] *= s, u[j] *= s;
  }
  vec o;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float v = g[j];
    if (GLU) v = unit_value(a.unit, g[j], u[j], a.limit, a.alpha);
    else if (a.unit == UNIT_RELU2) v = fmaxf(v, 0.f) * fmaxf(v, 0.f);
    o[j] = (T)v;
  }
  T* y = static_cast<T*>(a.y) + r * a.ldy + c;
  if (c + 4 <= a.ncol && a.ldy % 4 == 0) {
    *reinterpret_cast<vec*>(y) = o;
  } else {
    for (int j = 0; j < 4 && c + j < a.ncol; ++j) y[j] = o[j];
  }
}

// row of x that sorted row r reads
__device__ __forceinline__ const char* expert_row(const ExpertGemm& a, int r, int es) {
  return static_cast<const char*>(a.x) + (a.top > 0 ? a.src[r] / a.top : r) * a.ldx * es;
}

// (tile, column block) of this block among `cols` column blocks, or false.  Groups of four neighbouring tiles -- mostly one expert's --
// take all column blocks in turn on one XCD, so that their W panels and token rows meet in its L2, and go round the XCDs: a busy
// expert's groups, which share their panels, and those of the small ones, which stream them, spread over all memory paths (64
// experts of 512 x 1024, 700 tokens most of which go to 8: runs of neighbouring groups per XCD 75 us, dealt round 68).  What is left
// behind whole rounds of groups is dealt by equal runs: 16 tiles of 256 rows by 16 column blocks would run on four XCDs.  Small
// tiles come last, the same way.
__device__ __forceinline__ bool expert_place(const ExpertGemm& a, int cols, int& t, int& nb) {
  const int4 head = a.tiles[-1];
  int id = blockIdx.x, first = 0, live = head.y;
  if (id >= live * cols) {
    id -= live * cols;
    first = live;
    live = head.x - first;
    if (id >= live * cols) return false;
  }
  const int xcd = id & 7, k = id >> 3, rounds = live >> 5, dealt = rounds * 4 * cols;        // 32 tiles a round
  if (k < dealt) {
    const int grp = k / (4 * cols), in = k - grp * 4 * cols;
    t = first + (grp * 8 + xcd) * 4 + (in & 3);
    nb = in >> 2;
    return true;
  }
  const int left = live - 32 * rounds, nwg = left * cols, q = nwg >> 3, r = nwg & 7;
  id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k - dealt;
  const int grp = id / (4 * cols), in = id - grp * 4 * cols, gm = min(left - 4 * grp, 4);
  t = first + 32 * rounds + 4 * grp + in % gm;
  nb = in / gm;
  return true;
}

// ---- tile form ---------------------------------------------------------------------------------------------------
// WR row groups of W x MT tokens per block, 256 threads = 4 waves: 4 x 1 in blocks of 8 groups x 64 tokens, else 2 (W) x 2 (every other group
// of 16 tokens), a wave's sub-tile as FW x U accumulators (A = W: a lane's four registers are adjacent output columns).  A stage is 128
// bytes of K, ST of them in LDS: the W image keeps the pieces' order, the X image has rows of 128 B whose 16-B chunks are swizzled by
// (row / 2) % 8 (conflict-free b128 reads).  An expert's last tile is half full on average and with few rows its only one: groups of
// 16 tokens without a row are not multiplied (nor staged, with two stages), and the rest is dealt evenly over the waves.  f32 is bound by the matrix
// cores, whose work is a block's chain of 14 us (8 groups, K = 1024) for each 16 of its tokens: both products in us, every group multiplied / 8
// groups of W / 4 with three stages, 32 experts of 1024 x 512, buckets even and (spread by a factor of three): 338 tokens, top 4, 118 / 106 / 100
// (118 / 117 / 101), 800 180 / 168 / 158 (181 / 181 / 159), 520 119 / 119 / 104 (118 / 118 / 130), 1600 235 / 238 / 245 (236 / 235 / 243).  bf16 is
// bound by the way of the operands to LDS: 0 - 4 % shorter, and longer with blocks of 4 groups (1188 tokens of 2048 x 1024 145, 158) or a
// third stage (146 and 155 for 142 and 146).
template <typename T, int MT, int WR, int ST, bool GLU>
__global__ void __launch_bounds__(256, 163840 / (ST * (WR * 2048 + MT * 128))) expert_tile_kernel(ExpertGemm a) {
  constexpr int WIMG = WR * 2048, STG = WIMG + MT * 128, ES = sizeof(T);
  constexpr int WP = WR / 2, XP = MT / 32;     // 1-KiB pieces of the two images per wave
  constexpr int WB = MT == 64 && WR == 8 ? 1 : 2;             // waves over the tokens
  constexpr int FW = WR * WB / 4, U = MT / 16 / WB;           // a wave's row groups of W and of tokens
  __shared__ __attribute__((aligned(1024))) char smem[ST * STG];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (the half with the odd group of tokens in turn: a wave's place in its block is its SIMD)
  const int wa = w / WB, wb = WB == 1 ? 0 : (w ^ (blockIdx.x >> 3)) & 1, g = lane >> 4, col = lane & 15;
  int t, nb;
  if (!expert_place(a, (a.groups + WR - 1) / WR, t, nb)) return;
  const int4 tile = a.tiles[t];
  const int rows = __builtin_amdgcn_readfirstlane(tile.z), live = (rows + 15) / 16;

  const char* wsrc[WP];
#pragma unroll
  for (int i = 0; i < WP; ++i) {          // piece p = WP w + i of the stage: row group p / 2, K step p % 2
    const int p = WP * w + i;
    wsrc[i] = a.w + tile.x * a.wstride + ((long)min(nb * WR + p / 2, a.groups - 1) * a.kt + p % 2) * 1024 + lane * 16;
  }
  const char* xsrc[XP];
  int xoff[XP];
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int r = 8 * (4 * i + w) + lane / 8;
    xsrc[i] = expert_row(a, tile.y + min(r, rows - 1), ES);
    xoff[i] = 16 * ((lane % 8) ^ ((r >> 1) & 7));
  }
  const char* zero = reinterpret_cast<const char*>(&g_zero16);
  const unsigned lds0 = (unsigned)(uintptr_t)((__attribute__((address_space(3))) char*)smem);
  auto load = [&](const char* gp, unsigned dst) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(gp), "s"(dst)
                 : "memory");
  };
  const int ns = a.kt / 2;
  auto stage = [&](int s) {
    const unsigned buf = lds0 + (s % ST) * STG;
#pragma unroll
    for (int i = 0; i < WP; ++i) load(wsrc[i] + (long)s * 2048, buf + (WP * w + i) * 1024);
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      if (ST == 2 && 8 * (4 * i + w) >= 16 * live) break;
      const int off = s * 128 + xoff[i];
      load(off < a.kbytes ? xsrc[i] + off : zero, buf + WIMG + (4 * i + w) * 1024);
    }
  };
  f32x4 acc[FW][U];
#pragma unroll
  for (int f = 0; f < FW; ++f)
#pragma unroll
    for (int u = 0; u < U; ++u) acc[f][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < ST - 1; ++s)
    if (s < ns) stage(s);
  auto walk = [&](auto count) {           // all stages with this wave's first NU groups of tokens; every wave meets the same barriers
    constexpr int NU = decltype(count)::value;
    for (int s = 0; s < ns; ++s) {
      // this wave's pieces have landed, then everybody's; all reads of the other buffer are done
      if (ST == 2 || s + ST - 1 > ns) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 2) * (WP + XP)) : "memory");
      if (s + ST - 1 < ns) stage(s + ST - 1);
      const char* wi = smem + (s % ST) * STG + wa * FW * 2048 + lane * 16;
      const char* xi = smem + (s % ST) * STG + WIMG + (wb * 16 + col) * 128;
      uint4 av[FW][2], bv[NU][2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int f = 0; f < FW; ++f) av[f][kk] = *reinterpret_cast<const uint4*>(wi + (2 * f + kk) * 1024);
#pragma unroll
        for (int u = 0; u < NU; ++u)
          bv[u][kk] = *reinterpret_cast<const uint4*>(xi + u * WB * 2048 + (((4 * kk + g) ^ ((col >> 1) & 7)) << 4));
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
          for (int u = 0; u < NU; ++u) acc[f][u] = mma16<T>(av[f][kk], bv[u][kk], acc[f][u]);
    }
  };
  const int mine = (live - wb + WB - 1) / WB;   // (a wave of the second half may have none: it multiplies one that is not stored)
  if (U == 6 && mine >= 6) walk(Steps<U>{});
  else if (U == 6 && mine == 5) walk(Steps<U < 5 ? U : 5>{});
  else if (U >= 4 && mine >= 4) walk(Steps<U < 4 ? U : 4>{});
  else if (U >= 4 && mine == 3) walk(Steps<U < 3 ? U : 3>{});
  else if (mine >= 2) walk(Steps<2>{});
  else walk(Steps<1>{});
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int m = (u * WB + wb) * 16 + col;
    if (m >= rows) continue;
    const int G = nb * WR + wa * FW;
    if (GLU) {
#pragma unroll
      for (int q = 0; q < FW / 2; ++q)
        if (G + 2 * q < a.groups)
          expert_store<T, true>(a, tile.y + m, (G / 2 + q) * 16 + 4 * g, acc[2 * q][u], acc[2 * q + 1][u]);
    } else {
#pragma unroll
      for (int f = 0; f < FW; ++f)
        if (G + f < a.groups) expert_store<T, false>(a, tile.y + m, (G + f) * 16 + 4 * g, acc[f][u], acc[f][u]);
    }
  }
}

// ---- wide tile form (bf16) ---------------------------------------------------------------------------------------
// 256 W rows x 256 tokens per block, 8 waves as 2 (W rows) x 4 (tokens), a wave's 128 x 64 sub-tile as 8 x 4 accumulators:
// a third fewer operand reads per product than the 64 x 64 sub-tiles above, which are bound by them.  A K tile (64 elements) is
// four half tiles of 16 KiB -- W rows 0-63 of both wave rows, tokens 0-127, tokens 128-255, W rows 64-127 of both wave rows -- in
// two stages, and runs as four phases of {operand reads; one half tile of prefetch; barrier; 16 MFMAs; barrier}.  A half tile is
// staged again one phase after its last read, so three stay in flight across every barrier and the waits are counted, never a
// drain.  The waves of the second row run one barrier behind, so that a SIMD's two waves alternate between reading and
// multiplying.  A tile of at most 128 rows leaves out the products of the second half of its tokens.  One block per CU.
__device__ __forceinline__ void wide_bar() { __builtin_amdgcn_s_barrier(); }
template <int N> __device__ __forceinline__ void wide_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

template <bool GLU>
__global__ void __launch_bounds__(512) expert_wide_kernel(ExpertGemm a) {
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  union Frag {
    uint4 u;
    bf16x8 v;
  };
  constexpr int HALF = 16384, STG = 4 * HALF, W0 = 0, X0 = 1, X1 = 2, W1 = 3;
  __shared__ __attribute__((aligned(1024))) char smem[2 * STG];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wa = w >> 2, wb = w & 3, g = lane >> 4, col = lane & 15;
  int tl, nb;
  if (!expert_place(a, (a.groups + 15) / 16, tl, nb)) return;
  const int4 tile = a.tiles[tl];
  const int rows = tile.z;

  const char* src[4][2];                  // piece i of half tile h: this lane's 16 bytes of K tile 0
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int lr = 16 * w + 8 * i + (lane >> 3), ch = (lane & 7) ^ ((lr >> 1) & 7);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int G = min(nb * 16 + wa * 8 + wb + 4 * q, a.groups - 1);               // wave w stages row group w of the half
      src[q ? W1 : W0][i] = a.w + tile.x * a.wstride + ((long)G * a.kt + i) * 1024 + lane * 16;
      src[q ? X1 : X0][i] = expert_row(a, tile.y + min(128 * q + lr, rows - 1), 2) + 16 * ch;
    }
  }
  const unsigned lds0 = (unsigned)(uintptr_t)((__attribute__((address_space(3))) char*)smem);
  auto stage = [&](int h, int t, unsigned buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const unsigned dst = buf + h * HALF + (2 * w + i) * 1024;
      const char* gp = src[h][i] + (long)t * (h == W0 || h == W1 ? 2048 : 128);
      unsigned keep;
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep)
                   : "v"(gp), "s"(dst)
                   : "memory");
    }
  };
  const int rowoff = col * 128, ch0 = (g ^ ((col >> 1) & 7)) << 4, ch1 = ((4 + g) ^ ((col >> 1) & 7)) << 4;
  Frag av[4][2], b0[2][2], b1[2][2], c0[2][2];
  auto read_w = [&](const char* half) {
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        av[f][kk].u = *reinterpret_cast<const uint4*>(half + ((wa * 4 + f) * 2 + kk) * 1024 + lane * 16);
  };
  auto read_x = [&](const char* half, Frag (&b)[2][2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const char* r = half + (wb * 32 + t * 16) * 128 + rowoff;
      b[t][0].u = *reinterpret_cast<const uint4*>(r + ch0);
      b[t][1].u = *reinterpret_cast<const uint4*>(r + ch1);
    }
  };
  f32x4 acc[8][4];
#pragma unroll
  for (int f = 0; f < 8; ++f)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool second = rows > 128;
  auto phase = [&](auto F0c, auto T0c, const Frag (&bb)[2][2]) {
    constexpr int F0 = decltype(F0c)::value, T0 = decltype(T0c)::value;
    wide_bar();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (T0 == 0 || second) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            acc[F0 + f][T0 + t] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[f][kk].v, bb[t][kk].v, acc[F0 + f][T0 + t], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    wide_bar();
  };
  const int nt = a.kt / 2;
#pragma unroll
  for (int h = 0; h < 4; ++h) stage(h, 0, lds0);
  if (nt > 1) {
#pragma unroll
    for (int h = 0; h < 3; ++h) stage(h, 1, lds0 + STG);
    wide_wait<6>();
  } else {
    wide_wait<0>();
  }
  wide_bar();
  // The second wave row's extra barrier (the first row passes it after the loop).  A W half is staged again by the wave row that
  // reads it; an X half by the other row at least one barrier after this row's reads of it have returned (lgkmcnt(0) before the
  // row's next barrier); the counted wait of a K tile's last phase precedes both rows' barriers before the next tile's reads.
  if (wa == 1) wide_bar();
  auto ktile = [&](int t, Frag (&bc)[2][2], Frag (&bn)[2][2]) {
    const char* cur = smem + (t & 1) * STG;
    const char* nx = smem + ((t + 1) & 1) * STG;
    const unsigned lcur = lds0 + (t & 1) * STG, lnxt = lds0 + ((t + 1) & 1) * STG;
    const bool more1 = t + 1 < nt, more2 = t + 2 < nt;
    read_w(cur + W0 * HALF);
    if (more1) stage(W1, t + 1, lnxt);
    phase(Steps<0>{}, Steps<0>{}, bc);
    read_x(cur + X1 * HALF, b1);
    if (more2) stage(W0, t + 2, lcur);
    phase(Steps<0>{}, Steps<2>{}, b1);
    read_w(cur + W1 * HALF);
    if (more2) {
      stage(X0, t + 2, lcur);
      wide_wait<8>();                     // W0 and X0 of tile t + 1 have landed: four younger half tiles may be in flight
    } else {
      wide_wait<0>();
    }
    phase(Steps<4>{}, Steps<2>{}, b1);
    if (more1) read_x(nx + X0 * HALF, bn);
    if (more2) {
      stage(X1, t + 2, lcur);
      wide_wait<6>();                     // tile t + 1 whole
    } else {
      wide_wait<0>();
    }
    phase(Steps<4>{}, Steps<0>{}, bc);
  };
  read_x(smem + X0 * HALF, b0);
  int t = 0;
  for (; t + 1 < nt; t += 2) {
    ktile(t, b0, c0);
    ktile(t + 1, c0, b0);
  }
  if (t < nt) ktile(t, b0, c0);
  if (wa == 0) wide_bar();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int m = (u >> 1) * 128 + wb * 32 + (u & 1) * 16 + col, G = nb * 16 + wa * 8;
    if (m >= rows) continue;
    if (GLU) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (G + 2 * q < a.groups)
          expert_store<bf16, true>(a, tile.y + m, (G / 2 + q) * 16 + 4 * g, acc[2 * q][u], acc[2 * q + 1][u]);
    } else {
#pragma unroll
      for (int f = 0; f < 8; ++f)
        if (G + f < a.groups) expert_store<bf16, false>(a, tile.y + m, (G + f) * 16 + 4 * g, acc[f][u], acc[f][u]);
    }
  }
}

// ---- stream form -------------------------------------------------------------------------------------------------
// Up to 1024 pairs over up to 64 experts: every block finds its own tile (blockIdx.y) and the pairs in it, in the order of
// expert_plan_kernel, whose launch is left out; the first of a tile's blocks leaves the plan for the second product and the
// reader of its rows.  Bound by latency: one read of the indices and three passes through LDS, 1 - 3 us of the product for the 4 of the
// launch (passes of 1 - 64 rows with four such layers 1 - 13 us shorter: f32 1 row 592 / 583, 60 rows of width 1024 665 / 652, of 2048 1027 / 1020).
// own: the tile's pairs.  Returns (expert, first sorted row, rows, -).
template <int NW>
__device__ __forceinline__ int4 plan_tile(const ExpertGemm& a, int* own) {
  constexpr int THREADS = NW * 64, C = 1024 / THREADS;
  __shared__ int count[64], found[C][NW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, y = blockIdx.y, E = a.experts;
  const bool leave = blockIdx.x == 0;
  int held[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = threadIdx.x + THREADS * c;
    held[c] = i < a.pairs ? a.idx[i] : E;
  }
  if (threadIdx.x < 64) count[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < C; ++c)
    if ((unsigned)held[c] < (unsigned)E) atomicAdd(count + held[c], 1);
  __syncthreads();
  const int n = lane < E ? count[lane] : 0;
  int rows = n, upto = (n + 15) / 16;                        // this expert's and all before
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int r = __shfl_up(rows, o, 64), t = __shfl_up(upto, o, 64);
    if (lane >= o) rows += r, upto += t;
  }
  const unsigned long long past = __ballot(upto > y);
  int4 tile = make_int4(0, 0, 0, 0);
  int first = 0;                                             // of the tile among its expert's rows
  if (past != 0) {
    const int e = __ffsll(past) - 1, ne = __builtin_amdgcn_readlane(n, e);
    first = (y - (__builtin_amdgcn_readlane(upto, e) - (ne + 15) / 16)) * 16;
    tile = make_int4(e, __builtin_amdgcn_readlane(rows, e) - ne + first, min(16, ne - first), 0);
  }
  if (leave && threadIdx.x == 0) a.tiles_out[y] = tile;
  if (leave && y == 0)
#pragma unroll
    for (int c = 0; c < C; ++c)                              // identity entries have no row
      if (threadIdx.x + THREADS * c < a.pairs && (unsigned)held[c] >= (unsigned)E) a.pos[threadIdx.x + THREADS * c] = 0;
  if (tile.z == 0) return tile;
  int before[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const unsigned long long m = __ballot(held[c] == tile.x);
    before[c] = __popcll(m & ((1ull << lane) - 1));
    if (lane == 0) found[c][w] = __popcll(m);
  }
  __syncthreads();
  int at = -first;
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      const int r = at + before[c];
      if (v == w && held[c] == tile.x && r >= 0 && r < 16) {
        const int i = threadIdx.x + THREADS * c;
        own[r] = i;
        if (leave) {
          a.pos[i] = tile.y + r;
          a.src_out[tile.y + r] = i;
        }
      }
      at += found[c][v];
    }
  __syncthreads();
  return tile;
}

// Two row groups x 16 tokens per block; the NW waves share the four quarters of K, whose sums meet in LDS.  Bound by the weights' stream,
// past the caches as each is read once: four steps of weights and rows are always in flight per wave, and thin blocks of long streams
// keep many of them at it.  Both products in us, four groups x 4 waves that drain every eight steps (before) / the same drained never /
// two groups x 4 waves / two groups x 2 waves: 32 experts of 1024 x 2048, top 4, 1 token 19.5 / 15.9 / 15.9 / 15.8, 16 tokens 71 / 70 / 62 / 61, 64 tokens 80 /
// 79 / 70 / 70 (5.8 TB/s), f32 156 / 164 / 142 / 135; 8 of 2048 x 4096, 16 tokens 85 / 90 / 76 / 71; 16 of 512 x 1024, 8 tokens 17.3 / 14.8
// / 14.8 / 14.7.  Eight steps in flight measured the same.  Two waves have two quarters each, summed apart: the order of a row's sum, and with it
// its bits, must not follow from how many rows the step has.
template <typename T, bool GLU, bool PLAN, int NW>
__global__ void __launch_bounds__(NW * 64) expert_stream_kernel(ExpertGemm a) {
  constexpr int ES = sizeof(T), NF = 2, D = 4, QW = 4 / NW;
  __shared__ f32x4 red[4][NF][64];
  __shared__ int own[16];
  int4 tile;
  if constexpr (PLAN) tile = plan_tile<NW>(a, own);
  else tile = a.tiles[blockIdx.y];
  const int rows = tile.z;
  if (rows == 0) return;
  // (a wave's number of steps has to be uniform to the compiler: matrix instructions run whatever the lanes' mask)
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, col = lane & 15;
  const int G = blockIdx.x * NF;
  const int k0 = a.kt * w / NW, steps = a.kt * (w + 1) / NW - k0;
  const int mid = QW == 2 ? a.kt * (2 * w + 1) / 4 - k0 : 0;  // the wave's second quarter begins
  const char* wp[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f)
    wp[f] = reinterpret_cast<const char*>(a.w) + (tile.x * a.wstride + (long)min(G + f, a.groups - 1) * a.kt * 1024 + k0 * 1024) + 16 * lane;
  const char* xp = (PLAN ? static_cast<const char*>(a.x) + own[min(col, rows - 1)] / a.top * a.ldx * ES
                         : expert_row(a, tile.y + min(col, rows - 1), ES)) + 16 * g + k0 * 64;
  const int behind = a.kbytes - 16 * g - k0 * 64;            // the row's bytes from this lane's first chunk on
  const char* zero = reinterpret_cast<const char*>(&g_zero16);
  f32x4 acc[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  uint4 av[D][NF], bv[D];
  auto fetch = [&](int d, int k) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp[f] + k * 1024));
      av[d][f] = make_uint4(v.x, v.y, v.z, v.w);
    }
    bv[d] = *reinterpret_cast<const uint4*>(k * 64 < behind ? xp + k * 64 : zero);
  };
  auto first = [&] {                                         // quarter done: its sum aside
#pragma unroll
    for (int f = 0; f < NF; ++f) red[QW * w][f][lane] = acc[f], acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto use = [&](int d, int k) {
    if (QW == 2 && k == mid) first();
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = mma16<T>(av[d][f], bv[d], acc[f]);
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < steps) fetch(d, d);
  int k = 0;
  for (; k + 2 * D <= steps; k += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      use(d, k + d);
      fetch(d, k + D + d);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  for (; k < steps; k += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (k + d < steps) use(d, k + d);
      if (k + D + d < steps) fetch(d, k + D + d);
    }
  }
  if (QW == 2 && mid >= steps) first();
#pragma unroll
  for (int f = 0; f < NF; ++f) red[QW * w + QW - 1][f][lane] = acc[f];
  __syncthreads();
  auto total = [&](int i) {
    f32x4 s = red[0][i][lane];
#pragma unroll
    for (int v = 1; v < 4; ++v) s += red[v][i][lane];
    return s;
  };
  if (col >= rows) return;
  if (GLU) {
    if (w == 0 && G < a.groups) expert_store<T, true>(a, tile.y + col, G / 2 * 16 + 4 * g, total(0), total(1), PLAN ? own[col] : -1);
  } else if (w < NF && G + w < a.groups) {
    const f32x4 s = total(w);
    expert_store<T, false>(a, tile.y + col, (G + w) * 16 + 4 * g, s, s);
  }
}

// Tokens per tile, from the rows an expert gets on average.  A tile of 16 streams the weights once per 16 rows, a wider
// one wastes matrix work on rows that are not there but reads them once.  Both products, width 2048, 32 experts of 1024,
// bf16 (us, tiles of 16 / 64 / 128): 8 rows on average 81 / 84 / 87, 12: 86 / 85 / 87, 24: 118 / 87 / 89, 48: 172 / 90 /
// 96, 64: 209 / 127 / 98, 192: - / 183 / 148, 512: - / 355 / 320.  f32 products are bound by the matrix cores much
// earlier and gain nothing from 128 rows (width 1024, experts of 512): 8: 47 / 69, 24: 68 / 71, 32: 83 / 71 / 119,
// 96: 161 / 123 / 126, 512: - / 505 / 549.
//
// Beyond the line to wider tiles a few experts' column blocks may leave the chip idle, and a block's chain of stages, of about
// 1 us each and more with larger matrices, then takes longer than the weights streamed once per 16 rows by many small blocks.
// Both are estimated (us; `bytes`: an expert's two matrices; `stages`: of one block of each product): 4 experts of 4096 x 2048,
// tiles of 16 / 64: 32 rows on average 58 / 132, f32 126 / 569, 96 rows 120 / 122; 8 of 8192 x 2048: 24 rows 165 / 238, 48 rows
// 274 / 245; 2 of 4096 x 1024: 64 rows 32 / 87; 16 of 768 x 2048: 24 rows 35 / 48, 48 rows 56 / 50.
//
// Among the larger tiles the choice is by an estimate too: the rounds of blocks over the CUs (3, 2, 2 and 1 blocks of 64, 128, 192 and 256
// rows on each) times a block's stages at 1.35 (1.15 where the CUs are not full), 1.38, 1.84 and 1.85 us; an expert's last tile is half
// full on average, and a small one of 256 rows takes half the time.  Us for tiles of 64 / 128 / 256, bf16, experts' rows spread by a
// factor of about 1.3 (5 for the second figures): 32 experts of 1024 x 2048: 64 rows on average 102 / 100 / 95 (96 / 127 / 117), 128:
// 129 / 138 / 114 (132 / 139 / 142),
// 192: 165 / 146 / 156 (168 / 142 / 147), 256: 202 / 192 / 176 (189 / 188 / 174), 431: 290 / 256 / 245 (271 / 250 / 214), 633: 397 / 360 /
// 307 (371 / 325 / 298), 1024: 586 / 513 / 457 (570 / 505 / 447); of 512 x 1024: 128: 40 / 44 / 63, 256: 61 / 73 / 72, 431: 84 / 86 / 92,
// 633: 112 / 120 / 134; 8 of 2048 x 4096: 128: 145 / 136 / 144, 192: 197 / 138 / 157, 256: 204 / 216 / 167, 1250: 745 / 625 / 492; 64 of 768 x
// 2048: 64: 155 / 154 / 156, 128: 211 / 205 / 182, 512: 522 / 477 / 419; 4 plain ones of 4096 x 2048: 175: 67 / 79 / 68, 375: 95 / 92 / 142,
// 1000: 179 / 202 / 189.
struct Product {
  int groups, kt;
};

double wide_time(double avg, int experts, int mt, const Product* p) {
  double us = 0;
  for (int i = 0; i < 2; ++i) {
    const int cols = mt == 256 ? (p[i].groups + 15) / 16 : (p[i].groups + 7) / 8;
    double r = mt == 256 ? experts * (avg / 256 + 0.25) * cols / 256 + 0.2
                         : experts * (avg / mt + 0.5) * cols / (mt == 64 ? 768 : 512);
    if (r < 3) r = floor(r) + fmin(1.0, 2 * (r - floor(r)));      // the last of a few rounds leaves CUs idle
    us += fmax(r, 1.0) * (p[i].kt / 2 * (mt == 256 ? 1.85 : mt == 192 ? 1.84 : mt == 128 ? 1.38 : r < 1 ? 1.15 : 1.35) + (mt == 256 ? 5 : 0));
  }
  return us;
}

// `whole`: rows are whole stages of K, which the form of 256 rows asks for
int tile_rows(long pairs, int experts, int dt, const Product* p, bool whole) {
  const long avg = pairs / experts;
  if (avg <= (dt == 1 ? 24 : 12)) return 16;
  const double bytes = 1024.0 * ((double)p[0].groups * p[0].kt + (double)p[1].groups * p[1].kt);
  const int stages = (p[0].kt + p[1].kt) / 2;
  const double live = pairs < experts ? pairs : experts, memory = live * bytes / 5.2e6;
  const double chain = stages * (dt == 1 ? 1.15 + bytes * 20e-9 : 0.7 + bytes * 9.5e-9);
  const double again = (pairs / 16.0 + live / 2) * bytes / (dt == 1 ? 7.0e6 : 7.9e6);
  if (15 + (again > memory ? again : memory) < 12 + (chain > memory ? chain : memory) && pairs / 16 + experts <= 65535) return 16;
  if (dt == 1) return 64;
  const double t64 = wide_time((double)pairs / experts, experts, 64, p), t128 = wide_time((double)pairs / experts, experts, 128, p);
  // (below 512 rows an expert's panels are read by one or two blocks of 256, whose stages in flight do not cover a first touch of
  // memory: inside a model, 148 rows on average took 142 us with 256, 124 with 128, and 431 rows 254 and 246)
  if (whole && avg >= 512 && wide_time((double)pairs / experts, experts, 256, p) < fmin(t64, t128)) return 256;
  // 64 where it is clearly the shorter, and while most experts' only tile is less than half of one of 128: uneven buckets then pay for
  // the wider (plan and products, 200 and 300 tokens most of which go to an eighth of the experts: 64 of 512 x 1024, top 6, 128 rows 66 and 71 us,
  // 64 rows 47 and 51; 32 of 1024 x 2048, top 4, 120 and 126, 94 and 97; evenly spread 43 - 45 and 42, 91 - 92 and 86)
  // 192 takes a sixth less of the operands' way to LDS per row than 128, but its rounds are longer, and an expert with more rows than a tile starts
  // another of them: far beyond the 136 rows from which most experts fill more than one of 128 it has to be little worse by the
  // estimate, which is 5 - 10 % too low for two or three rounds of 128, else clearly better.  Us, 128 / 192 (even and spread buckets): 32 experts of 1024 x
  // 2048, 148 rows 142 / 145 (139 / 149), 192: 180 / 164 (180 / 164), 256: 190 / 175 (187 / 173), 338: 240 / 220 (234 / 216), 431: 265 / 250 (280 /
  // 252); of 512 x 1024, 256: 75 / 63, 432: 88 / 99, 633: 125 / 118; 64 of 768 x 2048, 141: 209 / 196 (201 / 187), 375: 372 / 340 (381 / 358);
  // 8 of 2048 x 4096, 150: 133 / 156, 250: 218 / 157 (211 / 157).
  const double t192 = wide_time((double)pairs / experts, experts, 192, p);
  if (avg >= 136 && t192 < (avg >= 176 ? 1.07 : 0.92) * fmin(t64, t128)) return 192;
  return avg <= 56 || t64 < 0.95 * t128 ? 64 : 128;
}

// f32 products in tiles of 64 tokens: four row groups of W a block, or eight (false)?  The matrix cores bound them, so what counts is how many
// blocks the fullest CU has, and halves even that out where whole ones leave a round of 256 up to half empty: `likely` tiles (an expert's last
// one half full) give x whole blocks a CU, of which halves cost half of ceil(2 x).  Both products in us, eight / four (three spreads of the buckets
// by three seeds each): 32 experts of 1024 x 512, 33 rows on average (x = 1.02) 77 / 75, 50 (1.28) 97 / 89, 65 (1.52) 115 / 107, but 80 (1.75) 114 /
// 127, 100 (2.06) 152 / 142, 120 (2.38) 177 / 155, 150 (2.84) 179 / 181; 8 of 2048 x 1024: 120 (1.19) 214 / 180, 200 (1.81) 217 / 245; 64 of 512 x 768
// 60 (4.31) 148 / 137; from 8 rounds on level.  The line at 0.65 is for the estimate, which is a tile or two off: over 55 such sets of both products
// 0.6 % and at most 5 % are lost to the better choice of each, with halves for all 1.2 % and 13 %, eight for all 4.2 % and 19 %.
bool half_blocks(double likely, int groups) {
  const double x = likely * ((groups + 7) / 8) / 256;
  return x < 8 && x - floor(x) <= 0.65;
}

template <typename T, bool GLU>
int expert_launch(const ExpertGemm& a, int mt, double likely, hipStream_t st) {
  if (mt == 256) {
    const long grid = (long)a.ntiles * ((a.groups + 15) / 16);
    if (grid > 0x7fffffff) return (int)hipErrorInvalidValue;
    if constexpr (sizeof(T) == 2) expert_wide_kernel<GLU><<<(unsigned)grid, 512, 0, st>>>(a);
  } else if (mt >= 64) {
    const long grid = (long)a.ntiles * ((a.groups + 7) / 8);
    if (grid > 0x7fffffff) return (int)hipErrorInvalidValue;
    if constexpr (sizeof(T) == 2) {
      if (mt == 192) expert_tile_kernel<T, 192, 8, 2, GLU><<<(unsigned)grid, 256, 0, st>>>(a);
      else if (mt == 128) expert_tile_kernel<T, 128, 8, 2, GLU><<<(unsigned)grid, 256, 0, st>>>(a);
      else expert_tile_kernel<T, 64, 8, 2, GLU><<<(unsigned)grid, 256, 0, st>>>(a);
    } else if (half_blocks(likely, a.groups)) {
      expert_tile_kernel<T, 64, 4, 3, GLU><<<(unsigned)(a.ntiles * ((a.groups + 3) / 4)), 256, 0, st>>>(a);
    } else {
      expert_tile_kernel<T, 64, 8, 2, GLU><<<(unsigned)grid, 256, 0, st>>>(a);
    }
  } else {
    if (a.ntiles > 65535) return (int)hipErrorInvalidValue;
    const dim3 grid((a.groups + 1) / 2, a.ntiles);
    // two waves a block where the blocks alone fill the chip, four otherwise (us of both products: above) and for the more rows of f32, whose
    // matrix work then counts (32 experts of 2048 x 2048, 24 rows each 531 with two, 510; 12 rows 317 and 313, 2 rows 240 and 245)
    const bool many = (long)a.ntiles * (a.groups / 4) >= 512 && a.pairs <= 12L * a.experts;
    if (a.idx != nullptr) {
      if (many) expert_stream_kernel<T, GLU, true, 2><<<grid, 128, 0, st>>>(a);
      else expert_stream_kernel<T, GLU, true, 4><<<grid, 256, 0, st>>>(a);
    } else if (many) expert_stream_kernel<T, GLU, false, 2><<<grid, 128, 0, st>>>(a);
    else expert_stream_kernel<T, GLU, false, 4><<<grid, 256, 0, st>>>(a);
  }
  return (int)hipGetLastError();
}

}  // namespace

// Rows of a tile (16: the stream form) that mx_experts takes for `pairs` over E experts with these products
MX_API int mx_experts_tile(int pairs, int E, int dt, int g1, int k1, int g2, int k2, int whole) {
  if (pairs < 1 || E < 1) return 0;
  const Product products[2] = {{g1, k1}, {g2, k2}};
  return tile_rows(pairs, E, dt, products, whole != 0 && pairs > 1024 && E <= 512);
}

// h [T, >= W] (row stride ldh), idx int32 [T, top] (>= E: an identity expert, no row here); w1 / w2: pieces as above, k1 / k2
// pieces per row group, g1 / g2 row groups per expert (gated units: g1 counts gate and up groups); unit: UNIT_*;
// scale f32 [T, top] on the experts' inputs (gated units) or null; act [T * top, lda], ys [T * top, W]: scratch of the
// storage type dt, lda >= F a multiple of 16 bytes; iws: ints, pos [T * top] | src
// [T * top] (each rounded up to 4) | tiles int4 [T * top / 16 + min(T * top, E) + 1]; afterwards pos is every pair's row of ys.
MX_API int mx_experts(const void* h, long ldh, const int* idx, int T, int top, int E, int W, int F, const void* w1, int k1,
                      int g1, const void* w2, int k2, int g2, int unit, float limit, float alpha, const float* scale,
                      void* act, long lda, void* ys, int* iws, int dt, hipStream_t st) {
  if (T <= 0) return 0;
  const int es = dt == 1 ? 4 : 2;
  const long P = (long)T * top;
  const bool glu = unit == UNIT_CLAMP || unit == UNIT_SILU || unit == UNIT_GELU;
  if (top < 1 || E < 1 || E > 8192 || P > 0x3fffffff || k1 % 2 || k2 % 2 || (long)k1 * 64 < (long)W * es || (long)k2 * 64 < lda * es ||
      lda < F || lda * es % 16 || (long)W * es % 16 || ldh * es % 16 || ((size_t)h | (size_t)act | (size_t)w1 | (size_t)w2) % 16 ||
      (size_t)iws % 16 || (glu ? g1 % 2 || g1 / 2 * 16 < lda : g1 * 16 < lda) || g2 * 16 < W || unit < 0 || unit > UNIT_RELU2 ||
      (scale != nullptr && !glu))
    return (int)hipErrorInvalidValue;
  // the plan by one block per expert beyond 1024 pairs (every block reads them all: up to 512 experts, 35 KB of counts)
  const bool wide = P > 1024 && E <= 512;
  const Product products[2] = {{g1, k1}, {g2, k2}};
  const int mt = tile_rows(P, E, dt, products, wide && (long)k1 * 64 == (long)W * es && (long)k2 * 64 == lda * es);
  const int ntiles = (int)(P / mt + (P < E ? P : E));
  int* pos = iws;
  int* src = iws + (P + 3) / 4 * 4;
  int4* tiles = reinterpret_cast<int4*>(src + (P + 3) / 4 * 4) + 1;
  int bits = 0;
  while ((1 << bits) < E) ++bits;
  int nw = (int)((P + 63) / 64);
  nw = nw < 1 ? 1 : (nw > 16 ? 16 : nw);
  while (nw > 1 && (long)(nw + 1) * E > 16384) --nw;         // counts per wave and the sums in 64 KB of LDS: 8192 experts
  const long run = (P + nw * 64 - 1) / (nw * 64);            // chunks of 64 pairs per wave
  const size_t lds = (size_t)(nw + 1) * E * 4;
#define PLAN(NC) expert_plan_kernel<NC><<<1, nw * 64, lds, st>>>(idx, (int)P, E, bits, mt, ntiles, pos, src, tiles)
#define WIDE(NC) expert_plan_wide_kernel<NC><<<E, 1024, (size_t)17 * E * 4, st>>>(idx, (int)P, E, mt, ntiles, pos, src, tiles)
  const bool own = mt == 16 && P <= 1024 && E <= 64;         // the first product's blocks plan for themselves
  if (own) {
  } else if (wide && P <= 4 * 1024) WIDE(4);
  else if (wide && P <= 8 * 1024) WIDE(8);
  else if (wide && P <= 16 * 1024) WIDE(16);
  else if (wide && P <= 32 * 1024) WIDE(32);
  else if (wide) WIDE(0);
  else if (run <= 2) PLAN(2);
  else if (run <= 8) PLAN(8);
  else if (run <= 16) PLAN(16);
  else if (run <= 32) PLAN(32);
  else PLAN(0);
#undef WIDE
#undef PLAN
  int rc = (int)hipGetLastError();
  if (rc) return rc;
  const double likely = (double)P / mt + 0.5 * (P < E ? P : E);
  ExpertGemm a{h, ldh, W * es, src, top, tiles, ntiles, (const char*)w1, (long)g1 * k1 * 1024, k1, g1, act, lda, (int)lda,
               unit, limit, alpha, scale, own ? idx : nullptr, (int)P, E, pos, src, tiles};
  ExpertGemm b{act, lda, (int)lda * es, src, 0, tiles, ntiles, (const char*)w2, (long)g2 * k2 * 1024, k2, g2, ys, W, W,
               UNIT_NONE, 0.f, 0.f, nullptr, nullptr, (int)P, E, nullptr, nullptr, nullptr};
  if (glu) MX_DISPATCH(dt, TT, rc = expert_launch<TT, true>(a, mt, likely, st));
  else MX_DISPATCH(dt, TT, rc = expert_launch<TT, false>(a, mt, likely, st));
  if (rc) return rc;
  MX_DISPATCH(dt, TT, rc = expert_launch<TT, false>(b, mt, likely, st));
  return rc;
}
