// Projections of a decode step of one to four rows: the weight once past the chip, and what surrounds a projection of a dense
// decoder layer in the same launch -- the RMS norm of its input before it, SiLU(gate) * up or the residual add behind it.
//
// At one row a layer of Llama-3-8B is 436 MB of weights, 75 us at the rate of a large copy; the split-K kernels
// (gemm_splitk.hip) with their separate norms, slab sums and reduce-SiLU pass take ten launches for it, of which the small
// ones last 3 - 5 us each whatever they do: 101 us with 26 of them beside the weights, 78 here, and
// the QKV form rotates and writes the cache as well (13.2 -> 10.7).  A workgroup owns 16 rows of W (a
// pair of gate and up groups) over all of K: its waves divide K, so no slabs, and each keeps 8 - 16 pieces of 1 KiB of W in flight
// in registers; the tokens' rows lie in LDS.  W's first pieces are issued before the norm waits for its row, so that the
// norm costs about its own latency once per launch.  Bound by the memory rate (5.9 TB/s for gate|up, 5.75 for the down
// projection), below 20 us by the launch and the way to memory as well.
// W: tile_weight's copy -- a piece is one A operand of the 16x16x32 matrix instruction -- and the tokens are its columns: one
// instruction per KiB of W whatever the number of rows.
#include "common.h"
#include "kv_layout.h"

namespace {

constexpr int FEW_ROWS = 4;              // tokens at most
constexpr int FEW_CHUNKS = 7168;         // 16-byte chunks of the rows at most: 4 x 14336, 3 x 18944, 2 x 28672, 1 x 57344 values in 112 KiB
constexpr int FEW_PAD = 64;              // bytes behind a token's row in LDS: four tokens at one k meet different banks

enum { FEW_SLAB = 0, FEW_ADD = 1, FEW_SILU = 2, FEW_ROPE = 3 };

struct FewRows {
  const bf16* x;                         // [M, K], row stride ldx
  const bf16* norm;                      // [K]: the rows are RMS-normed with it first; null: as they are
  const char* w;
  void* y;                               // f32 [M, N] | bf16 [M, N] += | bf16 [M, N / 2]
  long ldx, ldy;
  int M, N, K;
  float eps;
  // FEW_ROPE (heads of 128): y is q [M, Hq, 128]
  const int* positions;
  const float* cos_sin;                  // [positions, 128]: cos of 64 frequencies, then sin
  const int* slots;                      // of the paged cache; < 0: not written
  bf16* kc;
  bf16* vc;
  int Hq, Hkv;
};

// NORM: K <= 4096.  CHUNKS: the rows' 16-byte chunks, M * K / 8 at most; NW waves; DEPTH pieces of W in flight per wave.
template <int EPI, bool NORM, int CHUNKS, int NW, int DEPTH>
__global__ void __launch_bounds__(NW * 64) few_rows_kernel(FewRows a) {
  constexpr int XB = CHUNKS * 16 + FEW_ROWS * FEW_PAD;
  constexpr int GROUPS = EPI == FEW_SILU || EPI == FEW_ROPE ? 2 : 1, KW = NW / GROUPS, THREADS = NW * 64;
  __shared__ __attribute__((aligned(16))) char xs[XB];
  __shared__ f32x4 part[NW][64];
  __shared__ float sums[NW][FEW_ROWS];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, col = lane & 15;
  const int pitch = a.K * 2 + FEW_PAD, pieces = a.K / 32;
  // FEW_ROPE: a block owns the pairs of a rotation, row groups r and r + 4 of a head's eight
  const int group = EPI == FEW_ROPE ? (blockIdx.x >> 2) * 8 + (blockIdx.x & 3) + 4 * (w / KW) : blockIdx.x * GROUPS + w / KW;
  const int part_k = w % KW;
  const int p0 = pieces * part_k / KW, p1 = pieces * (part_k + 1) / KW;
  PENNY_DASSERT(a.M >= 1 && a.M <= FEW_ROWS && a.M * (a.K / 8) <= CHUNKS && group * 16 < a.N);

  // every load is issued without a branch, so that none waits for another: indices behind the end read the last chunk again
  constexpr int NC = !NORM ? 0 : THREADS < 512 ? 512 / THREADS : 1;   // NORM: chunks of a token per thread
  static_assert(CHUNKS % THREADS == 0, "every chunk has a thread");
  constexpr int XR = NORM ? FEW_ROWS * NC : CHUNKS / THREADS;
  const int kc = a.K / 8, all = a.M * kc, tid = threadIdx.x;
  uint4 xv[XR], nv[NORM ? NC : 1];
  auto row_of = [&](int i) { return (i >= kc) + (i >= 2 * kc) + (i >= 3 * kc); };
  if constexpr (NORM) {
#pragma unroll
    for (int m = 0; m < FEW_ROWS; ++m)
#pragma unroll
      for (int c = 0; c < NC; ++c)
        xv[m * NC + c] = reinterpret_cast<const uint4*>(a.x + min(m, a.M - 1) * a.ldx)[min(tid + THREADS * c, kc - 1)];
#pragma unroll
    for (int c = 0; c < NC; ++c) nv[c] = reinterpret_cast<const uint4*>(a.norm)[min(tid + THREADS * c, kc - 1)];
  } else {
#pragma unroll
    for (int c = 0; c < XR; ++c) {
      const int i = min(tid + THREADS * c, all - 1), m = row_of(i);
      xv[c] = reinterpret_cast<const uint4*>(a.x + m * a.ldx)[i - m * kc];
    }
  }
  const uint4* wp = reinterpret_cast<const uint4*>(a.w) + ((long)group * pieces + p0) * 64 + lane;
  const int np = p1 - p0;
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  auto piece = [&](int j) {              // read once and by nobody else: not kept in the caches
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp + (long)j * 64));
    return make_uint4(v[0], v[1], v[2], v[3]);
  };
  uint4 wv[DEPTH];
#pragma unroll
  for (int i = 0; i < DEPTH; ++i) wv[i] = piece(min(i, np - 1));

  if constexpr (NORM) {
#pragma unroll
    for (int m = 0; m < FEW_ROWS; ++m) {
      if (m >= a.M) break;
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        float v[8], t = 0.f;
        unpack8(xv[m * NC + c], v);
#pragma unroll
        for (int i = 0; i < 8; ++i) t += v[i] * v[i];
        ss += tid + THREADS * c < kc ? t : 0.f;
      }
      ss = wave_sum(ss);
      if (lane == 0) sums[w][m] = ss;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int m = 0; m < FEW_ROWS; ++m) {
      if (m >= a.M) break;
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < NW; ++i) ss += sums[i][m];
      const float inv = rsqrtf(ss / (float)a.K + a.eps);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        float v[8], n[8];
        unpack8(xv[m * NC + c], v);
        unpack8(nv[c], n);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (float)(bf16)(v[i] * inv) * n[i];   // the roundings of rmsnorm_kernel
        if (tid + THREADS * c < kc) *reinterpret_cast<uint4*>(xs + m * pitch + (tid + THREADS * c) * 16) = pack8(v);
      }
    }
  } else {
#pragma unroll
    for (int c = 0; c < XR; ++c) {
      const int i = tid + THREADS * c, m = row_of(i);
      if (i < all) *reinterpret_cast<uint4*>(xs + m * pitch + (i - m * kc) * 16) = xv[c];
    }
  }
  // the pieces of W stay in flight over the barrier: only LDS has to be complete
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  union Frag {
    uint4 u;
    bf16x8 v;
  };
  const char* xp = xs + min(col, a.M - 1) * pitch + p0 * 64 + g * 16;   // columns behind the last token repeat it and are dropped
  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
  auto multiply = [&](int i, int at) {
    Frag wf, xf;
    wf.u = wv[i];
    xf.u = *reinterpret_cast<const uint4*>(xp + at * 64);
    acc[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf.v, xf.v, acc[i & 1], 0, 0, 0);
  };
  int j = 0;
  for (; j + 2 * DEPTH <= np; j += DEPTH) {
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      multiply(i, j + i);
      wv[i] = piece(j + i + DEPTH);
    }
  }
  if (j + DEPTH < np) {
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      multiply(i, j + i);
      if (j + i + DEPTH < np) wv[i] = piece(j + i + DEPTH);
    }
    j += DEPTH;
  }
#pragma unroll
  for (int i = 0; i < DEPTH; ++i)
    if (j + i < np) multiply(i, j + i);
  part[w][lane] = acc[0] + acc[1];
  __syncthreads();
  if (w != 0 || col >= a.M) return;
  f32x4 sum[GROUPS];
#pragma unroll
  for (int s = 0; s < GROUPS; ++s) {
    sum[s] = part[s * KW][lane];
#pragma unroll
    for (int i = 1; i < KW; ++i) sum[s] += part[s * KW + i][lane];
  }
  if constexpr (EPI == FEW_ROPE) {         // as rope_kv_kernel with slabs: sums rounded to bf16, rotated in f32, rounded
    const int h = blockIdx.x >> 2, d = 16 * (blockIdx.x & 3) + 4 * g, slot = a.slots[col];
    float x1[4], x2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x1[i] = (float)(bf16)sum[0][i], x2[i] = (float)(bf16)sum[1][i];
    if (h < a.Hq + a.Hkv) {
      const float* cs = a.cos_sin + (long)a.positions[col] * 128 + d;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float co = cs[i], si = cs[64 + i], p = x1[i], q = x2[i];
        x1[i] = p * co - q * si;
        x2[i] = q * co + p * si;
      }
    }
    bf16x4 o1, o2;
#pragma unroll
    for (int i = 0; i < 4; ++i) o1[i] = (bf16)x1[i], o2[i] = (bf16)x2[i];
    const long blk = slot >= 0 ? slot / KV_BS : 0;
    const int off = slot >= 0 ? slot % KV_BS : 0;
    if (h < a.Hq) {
      bf16* dst = static_cast<bf16*>(a.y) + ((long)col * a.Hq + h) * 128 + d;
      *reinterpret_cast<bf16x4*>(dst) = o1;
      *reinterpret_cast<bf16x4*>(dst + 64) = o2;
    } else if (slot >= 0 && h < a.Hq + a.Hkv) {   // four adjacent channels lie in one 16-byte piece
      bf16* dst = a.kc + (blk * a.Hkv + h - a.Hq) * (long)(KV_BS * 128);
      *reinterpret_cast<bf16x4*>(dst + k_index(off, d, 128)) = o1;
      *reinterpret_cast<bf16x4*>(dst + k_index(off, d + 64, 128)) = o2;
    } else if (slot >= 0) {
      bf16* dst = a.vc + (blk * a.Hkv + h - a.Hq - a.Hkv) * (long)(KV_BS * 128);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dst[v_index(off, d + i, 128)] = o1[i];
        dst[v_index(off, d + 64 + i, 128)] = o2[i];
      }
    }
    return;
  }
  const int n = blockIdx.x * 16 + 4 * g;   // this lane's four adjacent outputs of token col
  if constexpr (EPI == FEW_SLAB) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + col * a.ldy + n) = sum[0];
  } else {
    bf16x4* y = reinterpret_cast<bf16x4*>(static_cast<bf16*>(a.y) + col * a.ldy + n);
    bf16x4 o;
    if constexpr (EPI == FEW_ADD) {
      const bf16x4 r = *y;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (bf16)((float)(bf16)sum[0][i] + (float)r[i]);   // as rmsnorm_kernel with slabs
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {                                              // as gemm_splitk.hip's SiLU epilogue
        const float gt = (float)(bf16)sum[0][i], up = (float)(bf16)sum[1][i];
        o[i] = (bf16)((float)(bf16)(gt / (1.f + __expf(-gt))) * up);
      }
    }
    *y = o;
  }
}

// Waves of a block and pieces in flight per wave, us of one row (four rows) on weights beyond the caches.  gate|up of 28672 x 4096: 8
// waves x 16 pieces 39.6 (40.3), 8 x 8 39.5 (40.6), 4 x 16 40.9 (40.2), 16 x 8 41.0 (45.7); QKV of 6144 x 4096: 8 x 12 10.4 (12.5), 8 x 16
// 11.3 (12.8), 4 x 16 11.2 (11.5); the adding form, 4096 x 14336: 16 x 8 20.4 (20.9), 8 x 24 21.0 (22.2), 4096 x 4096: 7.7 (8.4) and 9.1
// (9.8); QKV with its rotation and cache write behind it 16 x 8 10.7 (12.7), 16 x 12 11.3 (13.0), 8 x 16 13.8 (14.9), as two launches 13.2 (15.5).
// With loads that stay in the caches these were 42.3, 11.0, 22.8 and 8.5.
template <int EPI, bool NORM>
int launch_few(const FewRows& a, hipStream_t st) {
  const dim3 grid(a.N / (EPI == FEW_SILU || EPI == FEW_ROPE ? 32 : 16));
  constexpr int NW = EPI == FEW_ADD || EPI == FEW_ROPE ? 16 : 8, D = EPI == FEW_SILU ? 16 : EPI == FEW_SLAB ? 12 : 8;
  if (a.M * (a.K / 8) <= 2048) few_rows_kernel<EPI, NORM, 2048, NW, D><<<grid, NW * 64, 0, st>>>(a);
  else if constexpr (!NORM) few_rows_kernel<EPI, NORM, FEW_CHUNKS, NW, D><<<grid, NW * 64, 0, st>>>(a);
  return (int)hipGetLastError();
}

}  // namespace

// y = [norm of] X [M, K] x W [N, K]^T, W as tile_weight's copy.  form 0: norm, f32 [M, N]; 1: added to the bf16 rows of y in place;
// 2: norm, W is the interleave16 gate|up weight, y bf16 [M, N / 2] = SiLU(gate) * up.
// Contract (checked): 1 <= M <= 4, N % 16 == 0 (form 2: 32), K % 512 == 0, M * K <= 8 * FEW_CHUNKS; with a norm
// K <= 4096; ldx % 8 == 0, ldy % 4 == 0; x, norm, W and f32 y in whole 16 bytes, bf16 y in 8.
PENNY_API int penny_few_rows(const void* X, int ldx, const void* norm, float eps, const void* Wt, int K, int N, void* y, int ldy,
                             int M, int form, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > FEW_ROWS || N <= 0 || K <= 0 || N % (form == FEW_SILU ? 32 : 16) || K % 512 || ldx % 8 || ldy % 4 || form < 0 || form > 2 ||
      (long)M * K > 8 * FEW_CHUNKS || (form == FEW_ADD ? norm != nullptr : !norm || K > 4096) ||
      ((size_t)X | (size_t)norm | (size_t)Wt) % 16 || !X || !Wt || !y || (size_t)y % (form == FEW_SLAB ? 16 : 8))
    return (int)hipErrorInvalidValue;
  const FewRows a{(const bf16*)X, (const bf16*)norm, (const char*)Wt, y, ldx, ldy, M, N, K, eps};
  return form == FEW_SLAB ? launch_few<FEW_SLAB, true>(a, stream) : form == FEW_ADD ? launch_few<FEW_ADD, false>(a, stream) : launch_few<FEW_SILU, true>(a, stream);
}

// QKV [norm of] X [M, K] x W^T of heads of 128 with the rotation and the paged cache's write behind it (rope_kv.hip): q [M, Hq, 128] bf16,
// k and v of slots >= 0 into the caches.  W: tile_weight's copy of [(Hq + 2 Hkv) * 128, K].  Contract (checked): 1 <= M <= 4, K % 512 == 0,
// ldx % 8 == 0, a norm and K <= 4096; x, norm, W and the caches in whole 16 bytes.
PENNY_API int penny_few_qkv_rope(const void* X, int ldx, const void* norm, float eps, const void* Wt, int K, const int* positions,
                                 const float* cos_sin, const int* slots, void* q, void* kc, void* vc, int M, int Hq, int Hkv,
                                 hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > FEW_ROWS || !norm || K <= 0 || K % 512 || K > 4096 || ldx % 8 || Hq < 1 || Hkv < 1 || !positions || !cos_sin || !slots ||
      !X || !Wt || !q || !kc || !vc || ((size_t)X | (size_t)norm | (size_t)Wt | (size_t)q | (size_t)kc | (size_t)vc) % 16)
    return (int)hipErrorInvalidValue;
  FewRows a{(const bf16*)X, (const bf16*)norm, (const char*)Wt, q, ldx, 0, M, (Hq + 2 * Hkv) * 128, K, eps};
  a.positions = positions, a.cos_sin = cos_sin, a.slots = slots;
  a.kc = (bf16*)kc, a.vc = (bf16*)vc, a.Hq = Hq, a.Hkv = Hkv;
  return launch_few<FEW_ROPE, true>(a, stream);
}
