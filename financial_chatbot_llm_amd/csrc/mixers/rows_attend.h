// Softmax attention over paged cache rows on the matrix cores, shared by the windowed attention (a row holds the keys and
// values of its key/value heads) and the latent attention (a row is one latent: values are the first part of the keys).
//
// A block owns NW * MB * 16 (row, head) pairs of one segment and one key/value head -- QT consecutive rows x HB of its
// query heads -- and walks the tiles of KT keys that any of them sees.  Tiles are copied to LDS as they lie in the cache
// (LDS-DMA, two stages, one barrier per tile; 16-byte chunks swizzled by the row so that every operand read is free of
// bank conflicts).  Per tile and wave:
//     S^T = K Q^T     A: key rows from LDS, B: the wave's queries, in registers
//     softmax         base 2, the statistics of query lane % 16 live in that lane, f32; the running maximum moves only when
//                     a score exceeds it by 2^8; tiles that every pair sees whole skip the mask
//     O^T += V^T P^T  A: the value rows through the transposing LDS read (bf16) or element reads (f32), B: P straight from
//                     the score registers -- as two bf16 terms hi + lo, so that f32 weights are not cut to 8 bits (HILO), one
//                     bf16 term, or f32
// Bound by the LDS reads of the operands and the vector instructions of the softmax (four segments of 2048 rows, 16 heads
// over 4, window 1024: 127 us, 0.6 PFLOP/s with the second weight term).  Operands read a group ahead of their products, the page
// of a tile read a tile ahead of its copies and weights rounded in pairs took 4 - 7 % off in bf16 (prompts of 540, 300 and 327 rows
// behind 1000 - 2500 beside 21 rows: 70.2 -> 65.4 us) and 7 - 20 % in f32 (254 -> 228; latents, 2 single rows behind 1443: 42 -> 34).  16 pairs per wave (MB = 1): 32 halve the operand
// reads but leave two waves per SIMD (bf16 heads of 128: 56 against 43 us for 1190 rows) or spill (latent: 108 against 65).
// A block's serial walk is what a small step waits for: the caller splits the keys over nsplit blocks where that is shorter
// than reading the parts back (unnormalised: o | m | l, merged afterwards).
#pragma once
#include "mx_common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

struct RowsArgs {
  const void *q, *q2;            // queries: head h of row t at q + t * sq + h * D1 (elements), its second part at q2 + (t * H + h) * D2
  long sq;
  const void* cache;             // rows of Wr elements; kv head g: keys at g * kstep, values at voff + g * vstep
  int Wr, kstep, voff, vstep;
  const int *cu, *pos, *bt;
  int btw;
  const void* gate;              // [T, >= H] or, gate_elem, [T, >= H * P]; or null
  long sgate;
  int gate_elem, window, chunked, keep;
  const float* slope;            // [H] or null
  float cap;
  const float* sink;             // [H] or null
  float scale;
  void* out;                     // [T, H * P]
  int H, G, QT, HB;
  int S, per;                    // segments, row tiles of each (0: numbered by a scan)
  int nsplit;
  float* ws;                     // nsplit > 1: [T, H, nsplit, P + 2]
};

// 16 zero bytes: staged for keys behind a segment's last
__device__ uint4 g_rows_zero;

__device__ __forceinline__ float rows_max4(float v) {          // over the four lane groups
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float rows_sum4(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// chunk swizzle of a tile row (CH 16-byte chunks per row): chunk c lies at c ^ z(row).
// Rows of whole 256 bytes: 16 rows at one chunk (key reads) meet 16 different ones; bf16: rows 4 g .. 4 g + 7 at a pair of
// chunks (transposed value reads) different pairs; f32: rows 0, 4, 8, 12 at four chunks (value reads) different fours.
// 576-byte rows are 64 bytes apart in the banks by themselves: two bits do.  1152-byte rows (f32) are 128 bytes apart: three
// bits of the row pair; value reads then meet in pairs, which the f32 products they feed hide.
template <int CH, int ES> __device__ __forceinline__ int rows_swz(int row) {
  if (CH % 16 == 0) return ES == 2 ? ((row & 7) << 1) ^ ((row >> 3) & 1) : (((row >> 2) & 3) << 2) | (row & 3);
  if (CH % 8 == 0) return (row >> 1) & 7;
  return ((row >> 3) & 1) | ((row >> 1) & 2);
}

template <typename T, int D1, int D2, int P, bool SHARED, int MB, int NW, int KT, bool CAP, bool HILO>
__global__ void __launch_bounds__(NW * 64, NW == 4 ? 2 : 1) rows_attend_kernel(RowsArgs a) {
  constexpr int D = D1 + D2, ES = sizeof(T), KB = D * ES, VB = P * ES, KCH = KB / 16, VCH = VB / 16;
  constexpr int KIMG = KT * KB, STG = KIMG + (SHARED ? 0 : KT * VB);
  constexpr int KS = KB / 64, NT = P / 16, KTT = KT / 16, KI = KIMG / 1024, VI = SHARED ? 0 : KT * VB / 1024;
  constexpr int KPW = (KI + NW - 1) / NW, VPW = (VI + NW - 1) / NW;      // 1-KiB pieces per wave
  constexpr bool BF = ES == 2;
  // Two waves per SIMD or fewer (64 keys per tile, or f32) do not hide the LDS latency by themselves: operands are read a group
  // ahead of the products that use them.
  constexpr bool AHEAD = KT == 64 || !BF;
  constexpr int TP = BF && KS <= 4 ? 2 : 1, GK = BF ? KS : KS % 3 == 0 ? 3 : 2, GV = NT % 4 == 0 ? 4 : 1;
  constexpr int NVG = BF ? NT / GV : 4 * (NT / GV);
  static_assert(KTT % TP == 0 && KS % GK == 0, "operand groups");
  static_assert(KB % 64 == 0 && P % 16 == 0 && KIMG % 1024 == 0 && KT % 32 == 0 && PAGE_ROWS % KT == 0, "tile shape");
  __shared__ __attribute__((aligned(1024))) char smem[2 * STG];
  const int rep = a.H / a.G, hblocks = (rep + a.HB - 1) / a.HB;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const int split = blockIdx.x % a.nsplit;
  int s, t0;
  if (!mx_tile_place<4>(a.cu, a.S, a.per, a.QT, blockIdx.x / a.nsplit, s, t0)) return;
  const int r0 = a.cu[s], n = a.cu[s + 1] - r0;
  const int nq = min(a.QT, n - t0), kvh = blockIdx.y / hblocks, hg0 = (blockIdx.y % hblocks) * a.HB;
  const int nh = min(a.HB, rep - hg0), h0 = kvh * rep + hg0;
  const int p_first = a.pos[r0 + t0], p_last = a.pos[r0 + t0 + nq - 1];
  auto first_of = [&](int p) { return a.chunked ? (p / a.window) * a.window : max(0, p - a.window + 1); };
  const int lo = first_of(p_first), lo_last = first_of(p_last);

  // this lane's queries
  bool qok[MB];
  long row[MB];
  int hd[MB], pq[MB], pq_lo[MB];
  float slp[MB];
  uint4 qf[MB][KS];
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int pair = (w * MB + b) * 16 + c;
    qok[b] = pair < nq * nh;
    const int tq = qok[b] ? pair / nh : 0;
    row[b] = r0 + t0 + tq;
    hd[b] = h0 + (qok[b] ? pair - tq * nh : 0);
    pq[b] = qok[b] ? a.pos[row[b]] : -1;
    pq_lo[b] = qok[b] ? first_of(pq[b]) : 0;
    slp[b] = a.slope != nullptr ? a.slope[hd[b]] * 1.4426950408889634f : 0.f;
    const char* q1 = static_cast<const char*>(a.q) + (row[b] * a.sq + (long)hd[b] * D1) * ES;
    const char* q2 = static_cast<const char*>(a.q2) + (row[b] * a.H + hd[b]) * D2 * ES;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int o = 64 * k + 16 * g;
      qf[b][k] = *reinterpret_cast<const uint4*>(o < D1 * ES ? q1 + o : q2 + (o - D1 * ES));
    }
  }
  const bool wave_live = w * MB * 16 < nq * nh;
  f32x4 o[MB][NT];
  float m[MB], l[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    m[b] = -INFINITY;
    l[b] = 0.f;
#pragma unroll
    for (int i = 0; i < NT; ++i) o[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // tiles: nsink that hold kept first tokens and lie before the window's first one, then first_tile .. last
  const int first_tile = lo / KT, nsink = min((a.keep + KT - 1) / KT, first_tile);
  int ti = 0, t_end = nsink + p_last / KT - first_tile;          // walk indices, inclusive
  if (a.nsplit > 1) {
    const int per = (t_end + a.nsplit) / a.nsplit;
    ti = split * per;
    t_end = min(t_end, ti + per - 1);
  }
  auto key0 = [&](int i) { return (i < nsink ? i : first_tile + i - nsink) * KT; };

  // staging: piece i of a tile image is its i-th 1024 bytes, lane l its l-th 16
  int krow[KPW], koff[KPW], vrow[VPW > 0 ? VPW : 1], voff[VPW > 0 ? VPW : 1];
#pragma unroll
  for (int i = 0; i < KPW; ++i) {
    const int x = min(w + i * NW, KI - 1) * 64 + lane, r = x / KCH, ch = x % KCH;
    krow[i] = r;
    koff[i] = (r * a.Wr + kvh * a.kstep) * ES + ((ch ^ rows_swz<KCH, ES>(r)) << 4);
  }
#pragma unroll
  for (int i = 0; i < VPW; ++i) {
    const int x = min(w + i * NW, VI - 1) * 64 + lane, r = x / VCH, ch = x % VCH;
    vrow[i] = r;
    voff[i] = (r * a.Wr + a.voff + kvh * a.vstep) * ES + ((ch ^ rows_swz<VCH, ES>(r)) << 4);
  }
  const char* zero = reinterpret_cast<const char*>(&g_rows_zero);
  const unsigned lds0 = (unsigned)(uintptr_t)((__attribute__((address_space(3))) char*)smem);
  auto load = [&](const char* gp, unsigned dst) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(gp), "s"(dst)
                 : "memory");
  };
  auto page_of = [&](int i) { return a.bt[(long)s * a.btw + key0(i) / PAGE_ROWS]; };
  auto stage = [&](int i, int buf, int page) {
    const int k0 = key0(i), last = p_last - k0;
    const char* src = static_cast<const char*>(a.cache) +
                      ((long)__builtin_amdgcn_readfirstlane(page) * PAGE_ROWS + k0 % PAGE_ROWS) * a.Wr * ES;
    const unsigned dst = lds0 + buf * STG;
#pragma unroll
    for (int j = 0; j < KPW; ++j)
      if (KI % NW == 0 || w + j * NW < KI) load(krow[j] <= last ? src + koff[j] : zero, dst + (w + j * NW) * 1024);
#pragma unroll
    for (int j = 0; j < VPW; ++j)
      if (VI % NW == 0 || w + j * NW < VI) load(vrow[j] <= last ? src + voff[j] : zero, dst + KIMG + (w + j * NW) * 1024);
  };

  // operand addresses inside a stage
  const int zc = rows_swz<KCH, ES>(c);
  const int krd = c * KB;
  constexpr int VROWB = SHARED ? KB : VB, VC = SHARED ? KCH : VCH, VBASE = SHARED ? 0 : KIMG;
  const int vr = BF ? 4 * g + (c >> 2) : 4 * g;                  // first value row this lane reads
  const int zv = rows_swz<VC, ES>(vr);
  const float sl2 = a.scale * 1.4426950408889634f;
  const float cap_k = CAP ? 2.885390081777927f * a.scale / a.cap : 0.f;

  const int t_begin = ti;
  int buf = 0;
  // a tile's page is read a tile before its copies are issued, which would wait for it
  int page = ti < t_end ? page_of(ti + 1) : 0;
  if (ti <= t_end) stage(ti, 0, page_of(ti));
  for (; ti <= t_end; ++ti, buf ^= 1) {
    // this wave's pieces have landed, then everybody's; all reads of the other stage are done
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (ti < t_end) stage(ti + 1, buf ^ 1, page);
    if (ti + 1 < t_end) page = page_of(ti + 2);
    if (!wave_live) continue;
    const char* kt = smem + buf * STG;
    const int k0 = key0(ti);
    const bool whole = k0 + KT - 1 <= p_first && k0 >= lo_last;   // every pair sees every key
    f32x4 st[MB][KTT];
    uint4 kf[2][TP][GK];
    auto read_keys = [&](int i, uint4 (&f)[TP][GK]) {            // group i: TP key tiles of 16, GK steps of K
      const int t = i / (KS / GK) * TP, k = i % (KS / GK) * GK;
#pragma unroll
      for (int x = 0; x < TP; ++x)
#pragma unroll
        for (int y = 0; y < GK; ++y)
          f[x][y] = *reinterpret_cast<const uint4*>(kt + krd + (t + x) * 16 * KB + (((4 * (k + y) + g) ^ zc) << 4));
    };
#pragma unroll
    for (int t = 0; t < KTT; ++t)
#pragma unroll
      for (int b = 0; b < MB; ++b) st[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (AHEAD) read_keys(0, kf[0]);
#pragma unroll
    for (int i = 0; i < KTT / TP * (KS / GK); ++i) {
      if (!AHEAD) read_keys(i, kf[i & 1]);
      else if (i + 1 < KTT / TP * (KS / GK)) read_keys(i + 1, kf[(i + 1) & 1]);
      if (AHEAD) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int y = 0; y < GK; ++y)
#pragma unroll
        for (int x = 0; x < TP; ++x)
#pragma unroll
          for (int b = 0; b < MB; ++b) {
            const int t = i / (KS / GK) * TP + x, k = i % (KS / GK) * GK + y;
            st[b][t] = mma16<T>(kf[i & 1][x][y], qf[b][k], st[b][t]);
          }
      if (AHEAD) __builtin_amdgcn_sched_barrier(0);
    }
    // value operands, by groups of GV column tiles (f32: of one key step as well); the first group is on its way during the softmax
    const char* vt = kt + VBASE + vr * VROWB;
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    union VFrag {
      s16x4 s[2];
      bf16x8 v;
    };
    VFrag vb[2][GV][KTT / 2];
    float vf[2][GV][KTT];
    auto read_values = [&](int i) {
      if constexpr (BF) {
        const int cz = ((c & 3) >> 1) ^ zv, half = (c & 1) * 8;
#pragma unroll
        for (int x = 0; x < GV; ++x) {
          const char* v0 = vt + (((2 * (i * GV + x)) ^ cz) << 4) + half;
#pragma unroll
          for (int u = 0; u < KTT / 2; ++u) {
            VFrag& f = vb[i & 1][x][u];
            f.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(v0 + 32 * u * VROWB));
            f.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(v0 + (32 * u + 16) * VROWB));
          }
        }
      } else {
        // step (t, r): K index g is key 16 t + 4 g + r; the row's swizzle is that of row 4 g, but for its low two bits
        const int r = i / (NT / GV), i0 = i % (NT / GV) * GV;
#pragma unroll
        for (int x = 0; x < GV; ++x) {
          const char* v0 = vt + r * VROWB + (((4 * (i0 + x) + (c >> 2)) ^ rows_swz<VC, ES>(vr + r)) << 4) + (c & 3) * 4;
#pragma unroll
          for (int t = 0; t < KTT; ++t) vf[i & 1][x][t] = *reinterpret_cast<const float*>(v0 + 16 * t * VROWB);
        }
      }
    };
    if (AHEAD) {
      read_values(0);
      __builtin_amdgcn_sched_barrier(0);
    }
    union Pair {
      bf16x2 v;
      unsigned u;
    };
    union Weights {
      unsigned u[4];
      bf16x8 v;
    } ph[MB][KTT / 2], pl[MB][KTT / 2];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      float mt = -INFINITY;
      const float dist0 = (float)(k0 + 4 * g - pq[b]);           // j - p of this lane's first key
#pragma unroll
      for (int t = 0; t < KTT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float x;
          if (!CAP) x = st[b][t][r] * sl2;
          else if (BF) x = 1.4426950408889634f * (a.cap - 2.0f * a.cap * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(st[b][t][r] * cap_k)));
          else x = 1.4426950408889634f * a.cap * tanhf(st[b][t][r] * a.scale / a.cap);
          st[b][t][r] = x + slp[b] * (dist0 + (float)(16 * t + r));
        }
      if (!whole) {
#pragma unroll
        for (int t = 0; t < KTT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int j = k0 + 16 * t + 4 * g + r;
            st[b][t][r] = (j <= pq[b]) & ((j >= pq_lo[b]) | (j < a.keep)) ? st[b][t][r] : -INFINITY;
          }
      }
#pragma unroll
      for (int t = 0; t < KTT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) mt = fmaxf(mt, st[b][t][r]);
      mt = rows_max4(mt);
      const bool grow = mt > m[b] + 8.f;
      if (__any(grow)) {
        const float f = grow ? __builtin_amdgcn_exp2f(m[b] - mt) : 1.f;
        l[b] *= f;
#pragma unroll
        for (int i = 0; i < NT; ++i) o[b][i] *= f;
        m[b] = grow ? mt : m[b];
      }
      const float mref = m[b] == -INFINITY ? 0.f : m[b];
#pragma unroll
      for (int t = 0; t < KTT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          st[b][t][r] = __builtin_amdgcn_exp2f(st[b][t][r] - mref);
          l[b] += st[b][t][r];
        }
      if constexpr (BF) {
#pragma unroll
        for (int t = 0; t < KTT; ++t)
#pragma unroll
          for (int r = 0; r < 4; r += 2) {                       // by two: one conversion each
            const float p0 = st[b][t][r], p1 = st[b][t][r + 1];
            Pair hi, lo;
            hi.v = bf16x2{(bf16)p0, (bf16)p1};
            ph[b][t / 2].u[2 * (t & 1) + r / 2] = hi.u;
            if (HILO) {
              lo.v = bf16x2{(bf16)(p0 - __uint_as_float(hi.u << 16)), (bf16)(p1 - __uint_as_float(hi.u & 0xffff0000u))};
              pl[b][t / 2].u[2 * (t & 1) + r / 2] = lo.u;
            }
          }
      }
    }
#pragma unroll
    for (int i = 0; i < NVG; ++i) {
      if (!AHEAD) read_values(i);
      else if (i + 1 < NVG) read_values(i + 1);
      if (AHEAD) __builtin_amdgcn_sched_barrier(0);
      if constexpr (BF) {
#pragma unroll
        for (int u = 0; u < KTT / 2; ++u)
#pragma unroll
          for (int b = 0; b < MB; ++b) {
#pragma unroll
            for (int x = 0; x < GV; ++x)
              o[b][i * GV + x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb[i & 1][x][u].v, ph[b][u].v, o[b][i * GV + x], 0, 0, 0);
            if (HILO)
#pragma unroll
              for (int x = 0; x < GV; ++x)
                o[b][i * GV + x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb[i & 1][x][u].v, pl[b][u].v, o[b][i * GV + x], 0, 0, 0);
          }
      } else {
        const int r = i / (NT / GV), i0 = i % (NT / GV) * GV;
#pragma unroll
        for (int t = 0; t < KTT; ++t)
#pragma unroll
          for (int x = 0; x < GV; ++x)
#pragma unroll
            for (int b = 0; b < MB; ++b)
              o[b][i0 + x] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i & 1][x][t], st[b][t][r], o[b][i0 + x], 0, 0, 0);
      }
      if (AHEAD) __builtin_amdgcn_sched_barrier(0);
    }
  }
  typedef T out4 __attribute__((ext_vector_type(4)));
  const T* gate = static_cast<const T*>(a.gate);
  auto part_of = [&](long rw, int head) { return a.ws + ((rw * a.H + head) * a.nsplit + split) * (long)(P + 2); };
  auto out_of = [&](long rw, int head) { return static_cast<T*>(a.out) + (rw * a.H + head) * P; };
  auto gate_of = [&](long rw, int head) { return a.gate_elem ? gate + rw * a.sgate + (long)head * P : nullptr; };
  auto scale_of = [&](float mn, float lt, long rw, int head) {
    const float gs = mx_softmax_scale(mn, lt, a.sink, head);
    return gate != nullptr && !a.gate_elem ? gs * mx_sigmoid(ldf(gate + rw * a.sgate + head)) : gs;
  };
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    l[b] = rows_sum4(l[b]);
    // A key that a pair does not see has weight zero, but zero times a value that is not finite is not zero: pairs whose sums
    // came out so beside finite weights are walked again, by the whole wave, over the keys they see and no others.  (Looking
    // for them costs 0.2 - 0.4 us of bf16 calls of 17 - 300 us, up to 3 % in f32: 48 single rows 59.4 -> 61.5 us.)
    float zero_if_finite = 0.f;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) zero_if_finite = fmaf(o[b][i][r], 0.f, zero_if_finite);
    unsigned long long again = __ballot(zero_if_finite != 0.f && qok[b] && l[b] < INFINITY);
    again |= again >> 32;
    again = (again | again >> 16) & 0xffff;
    for (; again != 0; again &= again - 1) {
      const int at = __ffsll(again) - 1, head = __shfl(hd[b], at, 64), p = __shfl(pq[b], at, 64), p_lo = __shfl(pq_lo[b], at, 64);
      const long rw = r0 + t0 + ((w * MB + b) * 16 + at) / nh;
      const float sl = __shfl(slp[b], at, 64);
      const T* q1 = static_cast<const T*>(a.q) + rw * a.sq + (long)head * D1;
      const T* q2 = static_cast<const T*>(a.q2) + (rw * a.H + head) * D2;
      float wm = -INFINITY, wl = 0.f, acc[(P + 63) / 64] = {};
      for (int i = t_begin; i <= t_end; ++i) {
        const int k0 = key0(i);
        const T* tile = static_cast<const T*>(a.cache) +
                        ((long)a.bt[(long)s * a.btw + k0 / PAGE_ROWS] * PAGE_ROWS + k0 % PAGE_ROWS) * a.Wr;
        for (int j = k0; j < k0 + KT && j <= p; ++j) {
          if (j < p_lo && j >= a.keep) continue;
          const T* kr = tile + (long)(j - k0) * a.Wr + kvh * a.kstep;
          const T* vr = tile + (long)(j - k0) * a.Wr + a.voff + kvh * a.vstep;
          float x = 0.f;
          for (int d = lane; d < D; d += 64) x += ldf(d < D1 ? q1 + d : q2 + (d - D1)) * ldf(kr + d);
          x = mx_wave_sum(x) * a.scale;
          if (CAP) x = a.cap * tanhf(x / a.cap);
          x = x * 1.4426950408889634f + sl * (float)(j - p);
          const float mn = fmaxf(wm, x), f = __builtin_amdgcn_exp2f(wm - mn), wt = __builtin_amdgcn_exp2f(x - mn);
          wl = wl * f + wt;
          wm = mn;
#pragma unroll
          for (int u = 0; u < (P + 63) / 64; ++u)
            if (P % 64 == 0 || lane + 64 * u < P) acc[u] = acc[u] * f + wt * ldf(vr + lane + 64 * u);
        }
      }
      wm *= 0.6931471805599453f;
      const float gs = a.nsplit > 1 ? 1.f : scale_of(wm, wl, rw, head);
      const T* ge = gate_of(rw, head);
#pragma unroll
      for (int u = 0; u < (P + 63) / 64; ++u) {
        const int d = lane + 64 * u;
        if (P % 64 != 0 && d >= P) continue;
        if (a.nsplit > 1) part_of(rw, head)[d] = acc[u];
        else stf(out_of(rw, head) + d, acc[u] * gs * (ge != nullptr ? mx_sigmoid(ldf(ge + d)) : 1.f));
      }
      if (a.nsplit > 1 && lane < 2) part_of(rw, head)[P + lane] = lane == 0 ? wm : wl;
      if (c == at) qok[b] = false;                               // written
    }
    if (!qok[b]) continue;
    const float mn = m[b] * 0.6931471805599453f;                 // of the natural exponent
    if (a.nsplit > 1) {
      float* x = part_of(row[b], hd[b]);
      typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        *reinterpret_cast<f32x2*>(x + 16 * i + 4 * g) = f32x2{o[b][i][0], o[b][i][1]};
        *reinterpret_cast<f32x2*>(x + 16 * i + 4 * g + 2) = f32x2{o[b][i][2], o[b][i][3]};
      }
      if (g == 0) {
        x[P] = mn;
        x[P + 1] = l[b];
      }
      continue;
    }
    const float gs = scale_of(mn, l[b], row[b], hd[b]);
    T* dst = out_of(row[b], hd[b]) + 4 * g;
    const T* ge = a.gate_elem ? gate_of(row[b], hd[b]) + 4 * g : nullptr;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      out4 x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = (T)(o[b][i][r] * gs * (ge != nullptr ? mx_sigmoid(ldf(ge + 16 * i + r)) : 1.f));
      *reinterpret_cast<out4*>(dst + 16 * i) = x;
    }
  }
}

}  // namespace
