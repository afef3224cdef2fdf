// Backward of dense attention in fp32 on gfx950: contractions as split bf16 products (tpa_split3.h).
//
// Inputs are dense fp32 Q, K, V, dO [B, l, H, D], LSE [B, H, lq] (natural log) and
// delta = rowsum(O * dO) [B, H, lq]; outputs dense fp32 dQ, dK, dV.  With p = exp(x - lse):
//     dV = p^T dO,  dP = dO V^T,  dS = sm_scale * p * (dP - delta),  dQ = dS K,  dK = dS^T Q
// (tpa/tpa.py:546-995 computes the same quantities per block pair).  Two kernels, each of which
// owns its output rows and therefore needs no atomics:
//   bwd_f32_dq_kernel   workgroup = NW x 32 query rows of one head, loops over key tiles
//   bwd_f32_dkv_kernel  workgroup = NW x 32 keys of one head, loops over query tiles
// The operand placement is that of the fp32 forward kernel: the wave's own 32 rows (queries or
// keys) stay in registers, split, as B operands, so a lane holds the logits of ONE of its rows; the
// streamed tile (double buffered in LDS as three planes of bf16 parts per matrix) supplies the A operands in both
// roles - as rows (contraction over d) and read transposed (contraction over the tile's rows, in the order in which
// the accumulators hold them) - and p / dS are split in place as the B operands of the second contraction.
// Workgroups that meet values that do not split walk their tiles again with the fp32 instruction, which the kernels used
// to be made of.  Matrix cores and the vector work between the two contractions share the bound.  Whole backward, us, before
// and after: 2 x 2000 tokens, 64 heads of 64 causal 2459 / 1499, 4 x 4096, 16 heads of 128 8498 / 6727.
#include <type_traits>

#include "tpa_common.h"
#include "tpa_split3.h"

namespace tpa {
namespace {

struct BwdF32Params {
  const float *q, *k, *v, *d_o, *lse, *delta;
  const int32_t *qseg, *kvseg;
  float *dq, *dk, *dv;
  int B, lq, lk, H;
  float sm_scale;
  int causal, coff, nblk, npairs, groups;  // coff: with causal, row i sees keys <= i + coff; groups: see pair_of_workgroup
};

typedef std::integral_constant<bool, false> SplitProducts;
typedef std::integral_constant<bool, true> Fp32Products;

template <int D>
struct BwdLds {
  static constexpr int kTile = D == 128 ? 32 : 64;  // rows of the streamed tile: two buffers of six planes fit the LDS
  static constexpr int NMB = kTile / 32;
  static constexpr int RS = D + 16;                // row stride (bf16): row reads and transposed reads hit distinct banks
  static constexpr int kPlane = kTile * RS;
  static constexpr int kMat = 3 * kPlane;          // the parts h, m, l of one matrix
  // two matrices double buffered, then per buffer: lse2, delta, segment ids of the tile's rows
  static constexpr size_t kBytes = (size_t)4 * kMat * 2 + 2 * 3 * kTile * 4;
};

// The tile of dense X[b, row0 .., h, :] that `issue` fetched, into LDS; rows >= nrows as zeros.
template <int D, int NT>
struct TileRegs {
  static constexpr int CPR = D / 4, CH = BwdLds<D>::kTile * CPR / NT;
  f32x4 r[CH];
  __device__ __forceinline__ void issue(const float* base, int64_t row_stride, int row0, int nrows, bool scrub_nan) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int chunk = c * NT + threadIdx.x, t = chunk / CPR, cc = chunk % CPR;
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      if (row0 + t < nrows) x = *reinterpret_cast<const f32x4*>(base + (int64_t)(row0 + t) * row_stride + 4 * cc);
      if (scrub_nan) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = x[e] == x[e] ? x[e] : 0.f;
      }
      r[c] = x;
    }
  }
  // returns whether a value of this thread's does not split
  template <bool FP32>
  __device__ __forceinline__ bool store(uint16_t* dst, std::integral_constant<bool, FP32>) const {
    Magnitudes seen;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int chunk = c * NT + threadIdx.x, t = chunk / CPR, cc = chunk % CPR;
      uint16_t* const at = dst + t * BwdLds<D>::RS + 4 * cc;
      const f32x4& x = r[c];
      const Pair3 a = FP32 ? halves_of_pair(x[0], x[1]) : split_pair(x[0], x[1]), b = FP32 ? halves_of_pair(x[2], x[3]) : split_pair(x[2], x[3]);
      *reinterpret_cast<u32x2*>(at) = u32x2{a.h, b.h};
      *reinterpret_cast<u32x2*>(at + BwdLds<D>::kPlane) = u32x2{a.m, b.m};
      if constexpr (!FP32) {
        *reinterpret_cast<u32x2*>(at + 2 * BwdLds<D>::kPlane) = u32x2{a.l, b.l};
        seen.add(x);
      }
    }
    return seen.irregular();
  }
};

// The wave's own row, scaled and split (B operand of the row-wise contractions): lane (i, g) holds X[row][16 ks + 8 g + 0..7]
template <int D, bool FP32>
__device__ __forceinline__ bool load_own_row(const float* rowp, int g, float scale, bool scrub_nan, Split3 (&out)[D / 16], std::integral_constant<bool, FP32>) {
  Magnitudes seen;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    float y[8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(rowp + 16 * ks + 8 * g + 4 * u);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[4 * u + e] = (scrub_nan && x[e] != x[e] ? 0.f : x[e]) * scale;
    }
#pragma unroll
    for (int e = 0; e < 8; e += 2) seen.add(y[e], y[e + 1]);
    out[ks] = split8<FP32>(y);
  }
  return seen.irregular();
}

// The same as floats, split anew for every tile, for a wave whose registers do not hold both operands' parts.
template <int D>
struct OwnFloats {
  float x[D / 2];
  __device__ __forceinline__ bool load(const float* rowp, int g, float scale) {
    Magnitudes seen;
#pragma unroll
    for (int j = 0; j < D / 8; ++j) {
      const f32x4 y = *reinterpret_cast<const f32x4*>(rowp + 16 * (j >> 1) + 8 * g + 4 * (j & 1)) * scale;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * j + e] = y[e];
      seen.add(y);
    }
    return seen.irregular();
  }
};

// acc (rows of a 32-row block of the tile, lane = own row) = tile rows . own row, over d; `at`: the lane's place in the block
template <int D, bool FP32, typename Own>
__device__ __forceinline__ f32x16 rows_dot(const uint16_t* at, Own& own, std::integral_constant<bool, FP32>) {
  f32x16 acc, small;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = small[v] = 0.f;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    const uint16_t* const x = at + 16 * ks;
    const Split3 a = {*reinterpret_cast<const bf16x8*>(x), *reinterpret_cast<const bf16x8*>(x + BwdLds<D>::kPlane), *reinterpret_cast<const bf16x8*>(x + 2 * BwdLds<D>::kPlane)};
    if constexpr (std::is_same_v<Own, OwnFloats<D>>) {
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        asm volatile("" : "+a"(own.x[8 * ks + e]));  // keeps the parts from being formed ahead of the loop and held
        y[e] = own.x[8 * ks + e];
      }
      if constexpr (FP32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(join(a, e), y[e], acc, 0, 0, 0);
      } else {
        const Split3 b = split8(y);
        mfma_small(a, b, small);
        acc = mfma_bf16(a.h, b.h, acc);
      }
    } else if constexpr (FP32) {
      mfma_joined(a, own[ks], acc);
    } else {
      mfma_small(a, own[ks], small);
      acc = mfma_bf16(a.h, own[ks].h, acc);
    }
    if constexpr (D == 128) __builtin_amdgcn_sched_barrier(0);  // the operands of one step at a time: more do not fit the registers
  }
  if constexpr (!FP32)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] += small[v];
  return acc;
}

// out[db] (rows d = 32 db + accumulator row, lane = own row) += block^T . w, over the block's rows; w is an accumulator of
// rows_dot's layout (register v, half g <-> row 8 (v/4) + 4 g + v%4); `at`: the lane's place in the block (transposed)
template <int D, bool FP32>
__device__ __forceinline__ void cols_accumulate(const uint16_t* at, const f32x16& w, f32x16 (&out)[D / 32], std::integral_constant<bool, FP32>) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = w[8 * t + e];
    Split3 wf;
    if constexpr (!FP32) wf = split8(x);
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      bf16x8 part[3];
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) {
        const uint16_t* const y = at + pl * BwdLds<D>::kPlane + 16 * t * BwdLds<D>::RS + 32 * db;
        const s16x4 u0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)y);
        const s16x4 u1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(y + 8 * BwdLds<D>::RS));
        part[pl] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(u0, u1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
      const Split3 a = {part[0], part[1], part[2]};
      if constexpr (FP32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) out[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(join(a, e), x[e], out[db], 0, 0, 0);
      } else {
        mfma_small(a, wf, out[db]);
        out[db] = mfma_bf16(a.h, wf.h, out[db]);
      }
      if constexpr (D == 128) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <int D>
__device__ __forceinline__ void store_own_row(float* rowp, int g, const f32x16 (&acc)[D / 32]) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int vq = 0; vq < 4; ++vq)
      *reinterpret_cast<f32x4*>(rowp + 32 * db + 8 * vq + 4 * g) = f32x4{acc[db][4 * vq], acc[db][4 * vq + 1], acc[db][4 * vq + 2], acc[db][4 * vq + 3]};
}

template <int D>
__device__ __forceinline__ void clear(f32x16 (&acc)[D / 32]) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[db][v] = 0.f;
}

// ------------------------------------------------------------------------------------- dQ
template <int D, int NW, bool SEG>
__global__ __launch_bounds__(NW * 64) void bwd_f32_dq_kernel(BwdF32Params p) {
  typedef BwdLds<D> L;
  constexpr int NT = NW * 64, kBlock = NW * 32, kTile = L::kTile, NDB = D / 32, NKS = D / 16;
  extern __shared__ __attribute__((aligned(16))) float smem_bwd_f32[];
  uint16_t* const planes = reinterpret_cast<uint16_t*>(smem_bwd_f32);  // [2][K, V]
  int32_t* const lds_seg = reinterpret_cast<int32_t*>(planes + 4 * L::kMat);  // [2][kTile] key segment ids

  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int blk = p.nblk - 1 - pair / p.B;  // heaviest causal blocks first
  const int b = pair % p.B;
  const int tid = threadIdx.x, w = scalar(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
  const int q0 = blk * kBlock, wrow0 = q0 + 32 * w, qrow = wrow0 + i, qrow_ld = min(qrow, p.lq - 1);
  const int64_t hd = (int64_t)p.H * D;

  int kend = p.causal ? max(1, min(p.lk, q0 + kBlock + p.coff)) : p.lk, kbeg = 0;  // at least one (then fully masked) tile
  if constexpr (SEG) {  // only tiles that hold keys with ids of these rows
    int first, last;
    id_window<NT>(p.qseg + (int64_t)b * p.lq + q0, min(kBlock, p.lq - q0), p.kvseg + (int64_t)b * p.lk, kend, reinterpret_cast<int32_t*>(smem_bwd_f32), tid, first, last);
    kbeg = last < 0 ? 0 : first / kTile * kTile;
    kend = last < 0 ? 1 : last + 1;
  }
  const int ntiles = (kend - kbeg + kTile - 1) / kTile;
  const int wave_last_tile = p.causal ? min(ntiles - 1, max(wrow0 + p.coff + 31 - kbeg, 0) / kTile) : ntiles - 1;

  Split3 qf[NKS], gf[NKS];
  bool bad = false;
  auto load_own = [&](auto fp32, const auto& p, int row) __attribute__((always_inline)) {
    const int64_t at = ((int64_t)b * p.lq + row) * p.H * D + (int64_t)h * D;
    bad |= load_own_row<D>(p.q + at, g, p.sm_scale * kLog2e, false, qf, fp32);
    bad |= load_own_row<D>(p.d_o + at, g, 1.f, true, gf, fp32);
  };
  const float lse = p.lse[((int64_t)b * p.H + h) * p.lq + qrow_ld];
  // a row without a visible key (lse = -inf) has no gradient: +inf makes every p of the row zero
  const float lse2 = (qrow < p.lq && lse > -INFINITY) ? lse * kLog2e : INFINITY;
  const float delta = p.delta[((int64_t)b * p.H + h) * p.lq + qrow_ld];
  int32_t qseg = 0;
  if constexpr (SEG) qseg = p.qseg[(int64_t)b * p.lq + qrow_ld];
  const TileIds<SEG, 1> ids_of_wave({qseg});

  f32x16 dq[NDB];
  const float* const kbase = p.k + (int64_t)b * p.lk * hd + (int64_t)h * D;
  const float* const vbase = p.v + (int64_t)b * p.lk * hd + (int64_t)h * D;
  TileRegs<D, NT> kreg, vreg;
  int32_t seg_reg = 0;
  auto issue = [&](int tile) __attribute__((always_inline)) {
    kreg.issue(kbase, hd, kbeg + tile * kTile, kend, false);
    vreg.issue(vbase, hd, kbeg + tile * kTile, kend, false);
    if constexpr (SEG)
      if (tid < kTile) seg_reg = p.kvseg[(int64_t)b * p.lk + min(kbeg + tile * kTile + tid, p.lk - 1)];
  };
  auto commit = [&](auto fp32, int tile) __attribute__((always_inline)) {
    uint16_t* const at = planes + (tile & 1) * 2 * L::kMat;
    bad |= kreg.store(at, fp32);
    bad |= vreg.store(at + L::kMat, fp32);
    if constexpr (SEG)
      if (tid < kTile) lds_seg[(tile & 1) * kTile + tid] = seg_reg;
  };

  const int lp = l & 15, row_at = i * L::RS + 8 * g, col_at = (4 * g + (lp >> 2)) * L::RS + (l & 16) + 4 * (lp & 3);
  auto compute = [&](auto fp32, int tile) __attribute__((always_inline)) {
    const uint16_t* const ks = planes + (tile & 1) * 2 * L::kMat;
    const int k0 = kbeg + tile * kTile;
    const int limit = p.causal ? min(qrow + p.coff, kend - 1) : kend - 1;  // largest visible key index
#pragma unroll
    for (int mb = 0; mb < L::NMB; ++mb) {
      f32x16 s = rows_dot<D>(ks + 32 * mb * L::RS + row_at, qf, fp32);                      // x * log2(e)
      const f32x16 dp = rows_dot<D>(ks + L::kMat + 32 * mb * L::RS + row_at, gf, fp32);  // dP
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        int4 ids = {0, 0, 0, 0};
        if constexpr (SEG) ids = *reinterpret_cast<const int4*>(lds_seg + (tile & 1) * kTile + 32 * mb + 8 * vq + 4 * g);
        const int idv[4] = {ids.x, ids.y, ids.z, ids.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = 4 * vq + e, t = k0 + 32 * mb + 8 * vq + 4 * g + e;
          bool keep = t <= limit;
          if constexpr (SEG) keep = keep && idv[e] == qseg;
          const float pt = keep ? __builtin_amdgcn_exp2f(s[v] - lse2) : 0.f;
          s[v] = p.sm_scale * pt * (dp[v] - delta);  // dS
        }
      }
      if constexpr (!decltype(fp32)::value) bad |= too_large(s);
      cols_accumulate<D>(ks + 32 * mb * L::RS + col_at, s, dq, fp32);
    }
  };

  auto walk = [&](auto fp32) __attribute__((always_inline)) {
    clear<D>(dq);
    if constexpr (decltype(fp32)::value) load_own(fp32, *arguments_again<BwdF32Params>(), again(qrow_ld));
    else load_own(fp32, p, qrow_ld);
    issue(0);
    commit(fp32, 0);
    __syncthreads();
    for (int j = 0; j < ntiles; ++j) {
      const bool more = j + 1 < ntiles;
      if (more) issue(j + 1);
      if (j <= wave_last_tile && ids_of_wave.look(lds_seg + (j & 1) * kTile, l & (kTile - 1)) != kNoneOfThem) compute(fp32, j);
      if (more) commit(fp32, j + 1);
      __syncthreads();
    }
  };
  walk(SplitProducts{});
  if (__builtin_expect(__syncthreads_or(bad), 0)) walk(Fp32Products{});
  if (qrow < p.lq) store_own_row<D>(p.dq + ((int64_t)b * p.lq + qrow) * hd + (int64_t)h * D, g, dq);
}

// ------------------------------------------------------------------------------------- dK, dV
template <int D, int NW, bool SEG>
__global__ __launch_bounds__(NW * 64) void bwd_f32_dkv_kernel(BwdF32Params p) {
  typedef BwdLds<D> L;
  constexpr int NT = NW * 64, kBlock = NW * 32, kTile = L::kTile, NDB = D / 32, NKS = D / 16;
  extern __shared__ __attribute__((aligned(16))) float smem_bwd_f32[];
  uint16_t* const planes = reinterpret_cast<uint16_t*>(smem_bwd_f32);  // [2][Q, dO]
  float* const lds_row = reinterpret_cast<float*>(planes + 4 * L::kMat);  // [2][lse2 | delta | segment id][kTile]

  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int blk = pair / p.B;  // under the causal mask the first key blocks see the most rows: heaviest first
  const int b = pair % p.B;
  const int tid = threadIdx.x, w = scalar(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
  const int k0 = blk * kBlock, wkey0 = k0 + 32 * w, key = wkey0 + i, key_ld = min(key, p.lk - 1);
  const int64_t hd = (int64_t)p.H * D;

  // under the causal mask only rows at or after a key see it
  int first_tile = p.causal ? max(k0 - p.coff, 0) / kTile : 0;
  int ntiles = (p.lq + kTile - 1) / kTile;
  if constexpr (SEG) {  // only tiles that hold rows with ids of these keys
    int first, last;
    const int rbeg = min(first_tile * kTile, p.lq);
    id_window<NT>(p.kvseg + (int64_t)b * p.lk + k0, min(kBlock, p.lk - k0), p.qseg + (int64_t)b * p.lq + rbeg, p.lq - rbeg, reinterpret_cast<int32_t*>(smem_bwd_f32), tid, first, last);
    ntiles = last < 0 ? 0 : (rbeg + last) / kTile + 1;
    if (last >= 0) first_tile = (rbeg + first) / kTile;
  }
  const int wave_first_tile = p.causal ? max(wkey0 - p.coff, 0) / kTile : 0;

  std::conditional_t<D == 128, OwnFloats<D>, Split3[NKS]> kf, vf;
  bool bad = false;
  auto load_own = [&](auto fp32, const auto& p, int row) __attribute__((always_inline)) {
    const int64_t at = ((int64_t)b * p.lk + row) * p.H * D + (int64_t)h * D;
    if constexpr (D == 128) {  // with both accumulators the parts of both operands do not fit 512 registers
      bad |= kf.load(p.k + at, g, p.sm_scale * kLog2e);
      bad |= vf.load(p.v + at, g, 1.f);
    } else {
      bad |= load_own_row<D>(p.k + at, g, p.sm_scale * kLog2e, false, kf, fp32);
      bad |= load_own_row<D>(p.v + at, g, 1.f, false, vf, fp32);
    }
  };
  int32_t kseg = 0;
  if constexpr (SEG) kseg = p.kvseg[(int64_t)b * p.lk + key_ld];
  const TileIds<SEG, 1> ids_of_wave({kseg});

  f32x16 dk[NDB], dv[NDB];
  const float* const qbase = p.q + (int64_t)b * p.lq * hd + (int64_t)h * D;
  const float* const gbase = p.d_o + (int64_t)b * p.lq * hd + (int64_t)h * D;
  const float* const lse_b = p.lse + ((int64_t)b * p.H + h) * p.lq;
  const float* const delta_b = p.delta + ((int64_t)b * p.H + h) * p.lq;
  TileRegs<D, NT> qreg, greg;
  float row_reg = 0.f;  // threads 0 .. kTile - 1: lse2, then delta, then segment id of one row of the tile
  auto issue = [&](int tile) __attribute__((always_inline)) {
    qreg.issue(qbase, hd, tile * kTile, p.lq, false);
    greg.issue(gbase, hd, tile * kTile, p.lq, true);
    const int r = tile * kTile + (tid & (kTile - 1)), what = tid / kTile;
    if (what == 0) {
      const float lse = r < p.lq ? lse_b[r] : -INFINITY;
      row_reg = lse > -INFINITY ? lse * kLog2e : INFINITY;  // +inf: every p of the row is zero
    } else if (what == 1) {
      row_reg = r < p.lq ? delta_b[r] : 0.f;
    } else if (what == 2) {
      if constexpr (SEG) row_reg = __int_as_float(p.qseg[(int64_t)b * p.lq + min(r, p.lq - 1)]);
    }
  };
  auto commit = [&](auto fp32, int tile) __attribute__((always_inline)) {
    uint16_t* const at = planes + (tile & 1) * 2 * L::kMat;
    bad |= qreg.store(at, fp32);
    bad |= greg.store(at + L::kMat, fp32);
    if (tid < 3 * kTile) lds_row[(tile & 1) * 3 * kTile + tid] = row_reg;
  };

  const int lp = l & 15, row_at = i * L::RS + 8 * g, col_at = (4 * g + (lp >> 2)) * L::RS + (l & 16) + 4 * (lp & 3);
  auto compute = [&](auto fp32, int tile) __attribute__((always_inline)) {
    const uint16_t* const qs = planes + (tile & 1) * 2 * L::kMat;
    const float* const rows = lds_row + (tile & 1) * 3 * kTile;
    const int r0 = tile * kTile;
#pragma unroll
    for (int mb = 0; mb < L::NMB; ++mb) {
      f32x16 s = rows_dot<D>(qs + 32 * mb * L::RS + row_at, kf, fp32);              // x * log2(e); lane = key, registers = rows of the tile
      f32x16 dp = rows_dot<D>(qs + L::kMat + 32 * mb * L::RS + row_at, vf, fp32);  // dP
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const int off = 32 * mb + 8 * vq + 4 * g;
        const f32x4 lse2 = *reinterpret_cast<const f32x4*>(rows + off);
        const f32x4 dl = *reinterpret_cast<const f32x4*>(rows + kTile + off);
        f32x4 idf = {0.f, 0.f, 0.f, 0.f};
        if constexpr (SEG) idf = *reinterpret_cast<const f32x4*>(rows + 2 * kTile + off);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = 4 * vq + e, r = r0 + off + e;
          bool keep = !p.causal || key - p.coff <= r;
          if constexpr (SEG) keep = keep && __float_as_int(idf[e]) == kseg;
          const float pt = keep ? __builtin_amdgcn_exp2f(s[v] - lse2[e]) : 0.f;
          s[v] = pt;                                        // p
          dp[v] = p.sm_scale * pt * (dp[v] - dl[e]);        // dS
        }
      }
      if constexpr (!decltype(fp32)::value) bad |= too_large(s) | too_large(dp);
      cols_accumulate<D>(qs + L::kMat + 32 * mb * L::RS + col_at, s, dv, fp32);
      cols_accumulate<D>(qs + 32 * mb * L::RS + col_at, dp, dk, fp32);
    }
  };

  auto walk = [&](auto fp32) __attribute__((always_inline)) {
    clear<D>(dk);
    clear<D>(dv);
    if constexpr (decltype(fp32)::value) load_own(fp32, *arguments_again<BwdF32Params>(), again(key_ld));
    else load_own(fp32, p, key_ld);
    if (first_tile < ntiles) {
      issue(first_tile);
      commit(fp32, first_tile);
    }
    __syncthreads();
    for (int j = first_tile; j < ntiles; ++j) {
      const bool more = j + 1 < ntiles;
      if (more) issue(j + 1);
      bool mine = j >= wave_first_tile;
      if constexpr (SEG) mine = mine && ids_of_wave.look(reinterpret_cast<const int32_t*>(lds_row) + ((j & 1) * 3 + 2) * kTile, l & (kTile - 1)) != kNoneOfThem;
      if (mine) compute(fp32, j);
      if (more) commit(fp32, j + 1);
      __syncthreads();
    }
  };
  walk(SplitProducts{});
  if (__builtin_expect(__syncthreads_or(bad), 0)) walk(Fp32Products{});
  if (key < p.lk) {
    store_own_row<D>(p.dk + ((int64_t)b * p.lk + key) * hd + (int64_t)h * D, g, dk);
    store_own_row<D>(p.dv + ((int64_t)b * p.lk + key) * hd + (int64_t)h * D, g, dv);
  }
}

// ---------------------------------------------------------------------------------------------
// The same two kernels for problems with few blocks of 128 rows (or keys), whose launch leaves most of the chip idle and
// takes as long as one workgroup walking the whole sequence (`few_blocks` below).  A workgroup owns 32 rows (keys) and its
// NW waves split the streamed tiles, 32 rows each: wave w takes tiles w, w + NW, ... into LDS of its own (fp32, split on the
// way to the matrix cores; no barrier in the loop; the next tile's rows are in flight in registers meanwhile, one matrix at a
// time), and the partial sums are added through LDS in a fixed order.  What bounds them is one wave's chain of loads, LDS
// reads, splits and products: 2 x 1000 tokens, 8 heads of 64 causal, backward 114 us with the fp32 instruction, 98 so.
template <int D>
struct SplitLds {
  // eight waves where their tiles fit the LDS, as in the forward (tpa_prefill_f32.hip)
  static constexpr int NW = D == 64 ? 8 : 4;
  static constexpr int RS = D + 4;
  static constexpr int kMat = 32 * RS;
  static constexpr int kPerWave = 2 * kMat + 3 * 32;  // two matrices, then lse2 | delta | segment id of the tile's rows
  // the parts of one of the two own-row operands, which all waves read (registers hold the other)
  static constexpr int OS = D + 8, kOwnPlane = 32 * OS;
  static constexpr size_t kBytes = (size_t)NW * kPerWave * 4 + 3 * kOwnPlane * 2;
};

// 32 rows of dense X[b, row0 .., h, :] on their way to a wave's LDS; rows past the end read as zero
template <int D>
struct WaveTile {
  static constexpr int CPR = D / 4, RPI = 64 / CPR, NST = 32 / RPI;
  typedef f32x4 Regs[NST];
  __amdgpu_buffer_rsrc_t rs;
  int voff, row_bytes;
  __device__ __forceinline__ void describe(const float* base, int64_t hd, int nrows, int l) {
    rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, (int)(((int64_t)(nrows - 1) * hd + D) * 4), 0x00020000);
    voff = (int)(((l / CPR) * hd + 4 * (l % CPR)) * 4);
    row_bytes = (int)(hd * 4);
  }
  __device__ __forceinline__ void issue(int row0, Regs& r) const {
#pragma unroll
    for (int q = 0; q < NST; ++q)
      r[q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, (row0 + q * RPI) * row_bytes, 0));
  }
  // returns whether a value of this lane's does not split
  static __device__ __forceinline__ bool store(const Regs& r, float* dst, int l, bool scrub_nan) {
    Magnitudes seen;
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      f32x4 x = r[q];
      if (scrub_nan) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = x[e] == x[e] ? x[e] : 0.f;
      }
      seen.add(x);
      *reinterpret_cast<f32x4*>(dst + (q * RPI + l / CPR) * SplitLds<D>::RS + 4 * (l % CPR)) = x;
    }
    return seen.irregular();
  }
};

// The 32 own rows of one operand, scaled, split and parked for all waves; returns whether a value does not split
template <int D, bool FP32>
__device__ __forceinline__ bool park_own(const float* base, int64_t hd, int row0, int nrows, float scale, uint16_t* lds, int tid, std::integral_constant<bool, FP32>) {
  typedef SplitLds<D> L;
  constexpr int CPR = D / 4;
  Magnitudes seen;
  for (int idx = tid; idx < 32 * CPR; idx += L::NW * 64) {
    const int row = idx / CPR, cc = idx % CPR;
    const f32x4 x = *reinterpret_cast<const f32x4*>(base + (int64_t)min(row0 + row, nrows - 1) * hd + 4 * cc) * scale;
    seen.add(x);
    const Pair3 a = FP32 ? halves_of_pair(x[0], x[1]) : split_pair(x[0], x[1]), b = FP32 ? halves_of_pair(x[2], x[3]) : split_pair(x[2], x[3]);
    uint16_t* const at = lds + row * L::OS + 4 * cc;
    *reinterpret_cast<u32x2*>(at) = u32x2{a.h, b.h};
    *reinterpret_cast<u32x2*>(at + L::kOwnPlane) = u32x2{a.m, b.m};
    *reinterpret_cast<u32x2*>(at + 2 * L::kOwnPlane) = u32x2{a.l, b.l};
  }
  return seen.irregular();
}

// acc = tile rows . own row over d; `own(ks)` hands out the own row's operand of a step
template <int D, bool FP32, typename Own>
__device__ __forceinline__ f32x16 rows_dot32(const float* tile, int i, int g, Own&& own, std::integral_constant<bool, FP32>) {
  constexpr int RS = SplitLds<D>::RS;
  f32x16 acc, small;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = small[v] = 0.f;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    const Split3 o = own(ks);
    float x[8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const f32x4 f = *reinterpret_cast<const f32x4*>(tile + i * RS + 16 * ks + 8 * g + 4 * u);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * u + e] = f[e];
    }
    if constexpr (FP32) {
      Split3 b = o;
      asm volatile("" : "+v"(b.h), "+v"(b.m));  // not joined ahead of the loop (tpa_split3.h)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], join(b, e), acc, 0, 0, 0);
    } else {
      const Split3 a = split8(x);
      mfma_small(a, o, small);
      acc = mfma_bf16(a.h, o.h, acc);
      __builtin_amdgcn_sched_barrier(0);  // the operands of one step at a time: more do not fit the registers
    }
  }
  if constexpr (!FP32)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] += small[v];
  return acc;
}

// out[db] (rows d = (D/32) i + db, lane = own row) += tile^T . wgt over the tile's 32 rows
template <int D, bool FP32>
__device__ __forceinline__ void cols_accumulate32(const float* tile, int i, int g, const f32x16& wgt, f32x16 (&out)[D / 32], std::integral_constant<bool, FP32>) {
  constexpr int RS = SplitLds<D>::RS, NDB = D / 32;
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    float x[8], y[NDB][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = wgt[8 * t + e];
      const int v = 8 * t + e;
      const f32xN f = *reinterpret_cast<const f32xN*>(tile + (8 * (v >> 2) + 4 * g + (v & 3)) * RS + NDB * i);
#pragma unroll
      for (int db = 0; db < NDB; ++db) y[db][e] = f[db];
    }
    if constexpr (FP32) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int db = 0; db < NDB; ++db) out[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(y[db][e], x[e], out[db], 0, 0, 0);
    } else {
      const Split3 wf = split8(x);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        const Split3 a = split8(y[db]);
        mfma_small(a, wf, out[db]);
        out[db] = mfma_bf16(a.h, wf.h, out[db]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// a wave's accumulator as rows of 32 own rows x D in LDS
template <int D>
__device__ __forceinline__ void park(float* dst, int i, int g, const f32x16 (&acc)[D / 32]) {
  constexpr int NDB = D / 32;
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    f32xN out;
#pragma unroll
    for (int db = 0; db < NDB; ++db) out[db] = acc[db][v];
    *reinterpret_cast<f32xN*>(dst + i * SplitLds<D>::RS + NDB * (8 * (v >> 2) + 4 * g + (v & 3))) = out;
  }
}

// dst[row0 + r, h, :] = sum over the waves of what they parked at `at`
template <int D>
__device__ __forceinline__ void add_waves(const float* at, float* dst, int row0, int nrows, int64_t hd, int tid) {
  constexpr int CPR = D / 4, NW = SplitLds<D>::NW;
  for (int idx = tid; idx < 32 * CPR; idx += NW * 64) {
    const int r = idx / CPR, cc = idx % CPR;
    if (row0 + r >= nrows) break;
    f32x4 x = *reinterpret_cast<const f32x4*>(at + r * SplitLds<D>::RS + 4 * cc);
#pragma unroll
    for (int w = 1; w < NW; ++w) x += *reinterpret_cast<const f32x4*>(at + w * SplitLds<D>::kPerWave + r * SplitLds<D>::RS + 4 * cc);
    *reinterpret_cast<f32x4*>(dst + (int64_t)(row0 + r) * hd + 4 * cc) = x;
  }
}

template <int D, bool SEG>
__device__ __forceinline__ void dq_split(const BwdF32Params& p, int id) {
  typedef SplitLds<D> L;
  constexpr int NDB = D / 32, NKS = D / 16, NW = L::NW;
  extern __shared__ __attribute__((aligned(16))) float smem_bwd_f32[];
  int pair, h;
  if (!pair_of_workgroup(id, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int blk = p.nblk - 1 - pair / p.B, b = pair % p.B;  // heaviest causal blocks first
  const int tid = threadIdx.x, w = scalar(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
  const int q0 = blk * 32, qrow = q0 + i, qrow_ld = min(qrow, p.lq - 1);
  const int64_t hd = (int64_t)p.H * D;
  float* const lds_k = smem_bwd_f32 + w * SplitLds<D>::kPerWave;
  float* const lds_v = lds_k + SplitLds<D>::kMat;
  int32_t* const lds_seg = reinterpret_cast<int32_t*>(lds_v + SplitLds<D>::kMat);

  int kbeg = 0, kend = p.causal ? max(0, min(p.lk, q0 + 32 + p.coff)) : p.lk;
  int32_t qseg = 0;
  if constexpr (SEG) {
    qseg = p.qseg[(int64_t)b * p.lq + qrow_ld];
    int first, last;
    id_window<NW * 64>(p.qseg + (int64_t)b * p.lq + q0, min(32, p.lq - q0), p.kvseg + (int64_t)b * p.lk, kend, reinterpret_cast<int32_t*>(smem_bwd_f32), tid, first, last);
    kbeg = last < 0 ? 0 : first / 32 * 32;
    kend = last < 0 ? 0 : last + 1;
  }
  const int ntiles = (max(0, kend - kbeg) + 31) / 32;
  WaveTile<D> kt, vt;
  kt.describe(p.k + (int64_t)b * p.lk * hd + (int64_t)h * D, hd, max(kend, 1), l);
  vt.describe(p.v + (int64_t)b * p.lk * hd + (int64_t)h * D, hd, max(kend, 1), l);
  // one matrix is in flight at a time: V's tile is free after the first two products, K's after the third
  typename WaveTile<D>::Regs in;
  int32_t seg_in = 0;
  auto request_first = [&]() __attribute__((always_inline)) {
    if (w < ntiles) vt.issue(kbeg + 32 * w, in);
  };
  request_first();

  uint16_t* const lds_q = reinterpret_cast<uint16_t*>(smem_bwd_f32 + NW * L::kPerWave);
  Split3 gf[NKS];
  bool bad = false;
  auto load_own = [&](auto fp32) __attribute__((always_inline)) {
    bad |= park_own<D>(p.q + (int64_t)b * p.lq * hd + (int64_t)h * D, hd, q0, p.lq, p.sm_scale * kLog2e, lds_q, tid, fp32);
    bad |= load_own_row<D>(p.d_o + ((int64_t)b * p.lq + qrow_ld) * hd + (int64_t)h * D, g, 1.f, true, gf, fp32);
    __syncthreads();
  };
  load_own(SplitProducts{});
  int own_at = i * L::OS + 8 * g;
  auto q_operand = [&](int ks) __attribute__((always_inline)) -> Split3 {
    const uint16_t* const at = lds_q + own_at + 16 * ks;
    return {*reinterpret_cast<const bf16x8*>(at), *reinterpret_cast<const bf16x8*>(at + L::kOwnPlane), *reinterpret_cast<const bf16x8*>(at + 2 * L::kOwnPlane)};
  };
  auto g_operand = [&](int ks) __attribute__((always_inline)) -> const Split3& { return gf[ks]; };
  const float lse = p.lse[((int64_t)b * p.H + h) * p.lq + qrow_ld];
  // a row without a visible key (lse = -inf) has no gradient: +inf makes every p of the row zero
  const float lse2 = (qrow < p.lq && lse > -INFINITY) ? lse * kLog2e : INFINITY;
  const float delta = p.delta[((int64_t)b * p.H + h) * p.lq + qrow_ld];
  f32x16 dq[NDB];
  auto next_k = [&](int tile) __attribute__((always_inline)) {
    bad |= WaveTile<D>::store(in, lds_v, l, false);
    kt.issue(kbeg + 32 * tile, in);
    if constexpr (SEG) seg_in = p.kvseg[(int64_t)b * p.lk + min(kbeg + 32 * tile + i, p.lk - 1)];
  };
  auto arrive_k = [&]() __attribute__((always_inline)) {
    bad |= WaveTile<D>::store(in, lds_k, l, false);
    if constexpr (SEG) lds_seg[i] = seg_in;
  };
  auto walk = [&](auto fp32) __attribute__((always_inline)) {
    clear<D>(dq);
    if (w < ntiles) {
      next_k(w);
      arrive_k();
    }
    for (int tile = w; tile < ntiles; tile += NW) {
      const bool more = tile + NW < ntiles;
      if (more) vt.issue(kbeg + 32 * (tile + NW), in);
      const int k0 = kbeg + 32 * tile;
      asm volatile("" : "+v"(own_at));  // the operands in LDS are read again for every tile: held in registers they would not fit
      const f32x16 dp = rows_dot32<D>(lds_v, i, g, g_operand, fp32);
      f32x16 s = rows_dot32<D>(lds_k, i, g, q_operand, fp32);
      if (more) next_k(tile + NW);
      const int limit = p.causal ? min(qrow + p.coff, kend - 1) : kend - 1;  // largest visible key index
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        int4 ids = {0, 0, 0, 0};
        if constexpr (SEG) ids = *reinterpret_cast<const int4*>(lds_seg + 8 * vq + 4 * g);
        const int idv[4] = {ids.x, ids.y, ids.z, ids.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = 4 * vq + e;
          bool keep = k0 + 8 * vq + 4 * g + e <= limit;
          if constexpr (SEG) keep = keep && idv[e] == qseg;
          const float pt = keep ? __builtin_amdgcn_exp2f(s[v] - lse2) : 0.f;
          s[v] = p.sm_scale * pt * (dp[v] - delta);  // dS
        }
      }
      if constexpr (!decltype(fp32)::value) bad |= too_large(s);
      cols_accumulate32<D>(lds_k, i, g, s, dq, fp32);
      if (more) arrive_k();
    }
    park<D>(lds_k, i, g, dq);
  };
  walk(SplitProducts{});
  if (__builtin_expect(__syncthreads_or(bad), 0)) {
    request_first();
    load_own(Fp32Products{});
    walk(Fp32Products{});
    __syncthreads();
  }
  add_waves<D>(smem_bwd_f32, p.dq + (int64_t)b * p.lq * hd + (int64_t)h * D, q0, p.lq, hd, tid);
}

template <int D, bool SEG>
__device__ __forceinline__ void dkv_split(const BwdF32Params& p, int id) {
  typedef SplitLds<D> L;
  constexpr int NDB = D / 32, NKS = D / 16, NW = L::NW;
  extern __shared__ __attribute__((aligned(16))) float smem_bwd_f32[];
  int pair, h;
  if (!pair_of_workgroup(id, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int blk = pair / p.B, b = pair % p.B;  // under the causal mask the first key blocks see the most rows: heaviest first
  const int tid = threadIdx.x, w = scalar(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
  const int k0 = blk * 32, key = k0 + i, key_ld = min(key, p.lk - 1);
  const int64_t hd = (int64_t)p.H * D;
  float* const lds_q = smem_bwd_f32 + w * SplitLds<D>::kPerWave;
  float* const lds_g = lds_q + SplitLds<D>::kMat;
  float* const lds_row = lds_g + SplitLds<D>::kMat;  // [lse2 | delta | segment id][32]

  // under the causal mask only rows at or after a key see it
  int rbeg = p.causal ? min(p.lq, max(k0 - p.coff, 0)) / 32 * 32 : 0, rend = p.lq;
  int32_t kseg = 0;
  if constexpr (SEG) {
    kseg = p.kvseg[(int64_t)b * p.lk + key_ld];
    int first, last;
    id_window<NW * 64>(p.kvseg + (int64_t)b * p.lk + k0, min(32, p.lk - k0), p.qseg + (int64_t)b * p.lq + rbeg, p.lq - rbeg, reinterpret_cast<int32_t*>(smem_bwd_f32), tid, first, last);
    rend = last < 0 ? rbeg : rbeg + last + 1;
    if (last >= 0) rbeg = (rbeg + first) / 32 * 32;
  }
  const int ntiles = (max(0, rend - rbeg) + 31) / 32;
  const float* const lse_b = p.lse + ((int64_t)b * p.H + h) * p.lq;
  const float* const delta_b = p.delta + ((int64_t)b * p.H + h) * p.lq;
  WaveTile<D> qt, gt;
  qt.describe(p.q + (int64_t)b * p.lq * hd + (int64_t)h * D, hd, max(rend, 1), l);
  gt.describe(p.d_o + (int64_t)b * p.lq * hd + (int64_t)h * D, hd, max(rend, 1), l);
  // one matrix is in flight at a time: dO's tile is free after dV's product, Q's after dK's
  typename WaveTile<D>::Regs in;
  float row_in = 0.f;  // lanes 0-31: lse2, lanes 32-63: delta of one row of the tile
  int32_t seg_in = 0;
  auto request_first = [&]() __attribute__((always_inline)) {
    if (w < ntiles) gt.issue(rbeg + 32 * w, in);
  };
  request_first();
  bool bad = false;
  auto next_q = [&](int tile) __attribute__((always_inline)) {
    const int row0 = rbeg + 32 * tile, r = row0 + i;
    bad |= WaveTile<D>::store(in, lds_g, l, true);
    qt.issue(row0, in);
    const float x = (g ? delta_b : lse_b)[min(r, p.lq - 1)];
    // rows past the end and rows without a visible key (lse = -inf): +inf makes every p of the row zero
    row_in = g ? x : (r < rend && x > -INFINITY) ? x * kLog2e : INFINITY;
    if constexpr (SEG) seg_in = p.qseg[(int64_t)b * p.lq + min(r, p.lq - 1)];
  };
  auto arrive_q = [&]() __attribute__((always_inline)) {
    bad |= WaveTile<D>::store(in, lds_q, l, false);
    lds_row[l] = row_in;
    if constexpr (SEG) reinterpret_cast<int32_t*>(lds_row)[64 + i] = seg_in;
  };

  uint16_t* const lds_own = reinterpret_cast<uint16_t*>(smem_bwd_f32 + NW * L::kPerWave);
  Split3 vf[NKS];
  auto load_own = [&](auto fp32) __attribute__((always_inline)) {
    bad |= park_own<D>(p.k + (int64_t)b * p.lk * hd + (int64_t)h * D, hd, k0, p.lk, p.sm_scale * kLog2e, lds_own, tid, fp32);
    bad |= load_own_row<D>(p.v + ((int64_t)b * p.lk + key_ld) * hd + (int64_t)h * D, g, 1.f, false, vf, fp32);
    __syncthreads();
  };
  load_own(SplitProducts{});
  int own_at = i * L::OS + 8 * g;
  auto k_operand = [&](int ks) __attribute__((always_inline)) -> Split3 {
    const uint16_t* const at = lds_own + own_at + 16 * ks;
    return {*reinterpret_cast<const bf16x8*>(at), *reinterpret_cast<const bf16x8*>(at + L::kOwnPlane), *reinterpret_cast<const bf16x8*>(at + 2 * L::kOwnPlane)};
  };
  auto v_operand = [&](int ks) __attribute__((always_inline)) -> const Split3& { return vf[ks]; };
  f32x16 dk[NDB], dv[NDB];

  auto walk = [&](auto fp32) __attribute__((always_inline)) {
    clear<D>(dk);
    clear<D>(dv);
    if (w < ntiles) {
      next_q(w);
      arrive_q();
    }
    for (int tile = w; tile < ntiles; tile += NW) {
      const bool more = tile + NW < ntiles;
      if (more) gt.issue(rbeg + 32 * (tile + NW), in);
      const int r0 = rbeg + 32 * tile;
      asm volatile("" : "+v"(own_at));
      f32x16 dp = rows_dot32<D>(lds_g, i, g, v_operand, fp32);  // lane = key, registers = rows of the tile
      f32x16 s = rows_dot32<D>(lds_q, i, g, k_operand, fp32);
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const int off = 8 * vq + 4 * g;
        const f32x4 lse2 = *reinterpret_cast<const f32x4*>(lds_row + off);
        const f32x4 dl = *reinterpret_cast<const f32x4*>(lds_row + 32 + off);
        int4 ids = {0, 0, 0, 0};
        if constexpr (SEG) ids = *reinterpret_cast<const int4*>(lds_row + 64 + off);
        const int idv[4] = {ids.x, ids.y, ids.z, ids.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = 4 * vq + e;
          bool keep = !p.causal || key - p.coff <= r0 + off + e;
          if constexpr (SEG) keep = keep && idv[e] == kseg;
          const float pt = keep ? __builtin_amdgcn_exp2f(s[v] - lse2[e]) : 0.f;
          s[v] = pt;                                 // p
          dp[v] = p.sm_scale * pt * (dp[v] - dl[e]);  // dS
        }
      }
      if constexpr (!decltype(fp32)::value) bad |= too_large(s) | too_large(dp);
      cols_accumulate32<D>(lds_g, i, g, s, dv, fp32);
      if (more) next_q(tile + NW);
      cols_accumulate32<D>(lds_q, i, g, dp, dk, fp32);
      if (more) arrive_q();
    }
    park<D>(lds_q, i, g, dk);
    park<D>(lds_g, i, g, dv);
  };
  walk(SplitProducts{});
  if (__builtin_expect(__syncthreads_or(bad), 0)) {
    request_first();
    load_own(Fp32Products{});
    walk(Fp32Products{});
    __syncthreads();
  }
  add_waves<D>(smem_bwd_f32, p.dk + (int64_t)b * p.lk * hd + (int64_t)h * D, k0, p.lk, hd, tid);
  add_waves<D>(smem_bwd_f32 + SplitLds<D>::kMat, p.dv + (int64_t)b * p.lk * hd + (int64_t)h * D, k0, p.lk, hd, tid);
}

// Both in one launch: the dK/dV workgroups first (four products per tile against three), then the dQ ones, which fill the
// compute units that the tail of the first leaves idle: a launch and its gap less (2 x 1000 tokens, 8 heads of 64, whole
// training step 133.3 -> 131.3 us with the factors of the projections requested a rank ahead).
struct BwdF32Pair { BwdF32Params kv, q; int n_kv; };
template <int D, bool SEG>
__global__ __launch_bounds__(SplitLds<D>::NW * 64, 1) void bwd_f32_split_kernel(BwdF32Pair p) {
  if ((int)blockIdx.x < p.n_kv) dkv_split<D, SEG>(p.kv, blockIdx.x);
  else dq_split<D, SEG>(p.q, blockIdx.x - p.n_kv);
}

// Whether 32-row workgroups pay: the launch of 128-row ones leaves half of the 256 compute units idle, or fills them once
// with causal blocks of long sequences, of which the heaviest is twice the average.  Backward, us, 32 / 128 rows: 8 heads of
// 64, 2 x 1000 tokens causal 98 / 201, 4 x 1000 177 / 207, 8 x 1000 343 / 261, not causal 2 x 1000 143 / 205, 4 x 1000
// 270 / 217; 16 heads of 128 causal, 4 x 512 253 / 258, 8 x 256 194 / 166, 1 x 2000 555 / 788.  The split kernels' buffer
// offsets take a batch entry below 2 GiB.
bool few_blocks(const BwdF32Params& p, int rows, int D) {
  const int64_t big = p.lq > p.lk ? p.lq : p.lk;
  return (int64_t)((rows + 127) / 128) * p.B * p.H <= (p.causal && rows >= 512 ? 256 : 128) && (big + 64) * p.H * D * 4 < (int64_t(1) << 31);
}

// Head size 64: eight waves on blocks of 256 rows, two per SIMD, where those fill the chip.  Backward, us, eight / four waves,
// 8 heads: 4 x 4000 causal 1280 / 1483, 8 x 2000 733 / 831, 4 x 2000 (256 blocks, the heaviest twice the average)
// 569 / 427, 8 x 1000 not causal 359 / 411, 4 x 1000 308 / 217.  At head size 128 their registers do not hold the operands.
bool many_blocks(const BwdF32Params& p, int rows) { return (int64_t)((rows + 255) / 256) * p.B * p.H >= (p.causal ? 512 : 256); }

// fills in the decomposition of `rows` rows (or keys) in blocks of `block`; the number of workgroups
int64_t decompose(BwdF32Params& p, int rows, int block) {
  p.nblk = (rows + block - 1) / block;
  p.npairs = p.nblk * p.B;
  p.groups = head_groups(p.npairs, p.H);
  return workgroups_of(p.npairs, p.H, p.groups);
}

template <typename K>
int launch_kernel(K kern, bool (&configured)[kMaxDevices], int rows, int waves, size_t lds, BwdF32Params p, hipStream_t stream) {
  const int64_t n = decompose(p, rows, 32 * waves);
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), lds); rc != TPA_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3(64 * waves), lds, stream, p);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

template <int D, bool SEG>
int launch_split(const BwdF32Params& p, bool dq, bool dkv, hipStream_t stream) {
  static bool configured[kMaxDevices] = {};
  auto kern = bwd_f32_split_kernel<D, SEG>;
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), SplitLds<D>::kBytes); rc != TPA_OK) return rc;
  BwdF32Pair pair{p, p, 0};
  const int64_t nk = decompose(pair.kv, p.lk, 32), nq = decompose(pair.q, p.lq, 32);
  pair.n_kv = dkv ? (int)nk : 0;
  hipLaunchKernelGGL(kern, dim3((unsigned)(pair.n_kv + (dq ? nq : 0))), dim3(SplitLds<D>::NW * 64), SplitLds<D>::kBytes, stream, pair);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

template <int D, bool SEG>
int launch_pair(const BwdF32Params& p, hipStream_t stream) {
  static bool configured[4][kMaxDevices] = {};
  const bool split_dq = few_blocks(p, p.lq, D), split_dkv = few_blocks(p, p.lk, D);
  if (split_dq || split_dkv)
    if (int rc = launch_split<D, SEG>(p, split_dq, split_dkv, stream); rc != TPA_OK) return rc;
  int rc = TPA_OK;
  if (!split_dq) {
    if constexpr (D == 64) rc = many_blocks(p, p.lq) ? launch_kernel(bwd_f32_dq_kernel<D, 8, SEG>, configured[0], p.lq, 8, BwdLds<D>::kBytes, p, stream)
                                                     : launch_kernel(bwd_f32_dq_kernel<D, 4, SEG>, configured[1], p.lq, 4, BwdLds<D>::kBytes, p, stream);
    else rc = launch_kernel(bwd_f32_dq_kernel<D, 4, SEG>, configured[1], p.lq, 4, BwdLds<D>::kBytes, p, stream);
  }
  if (rc != TPA_OK || split_dkv) return rc;
  if constexpr (D == 64)
    if (many_blocks(p, p.lk)) return launch_kernel(bwd_f32_dkv_kernel<D, 8, SEG>, configured[2], p.lk, 8, BwdLds<D>::kBytes, p, stream);
  return launch_kernel(bwd_f32_dkv_kernel<D, 4, SEG>, configured[3], p.lk, 4, BwdLds<D>::kBytes, p, stream);
}

}  // namespace
}  // namespace tpa

// dense fp32 q, k, v, d_o [B, l, H, D] with D in {64, 128}, rows 16-byte aligned, no bias
int dense_bwd_f32_supported(int dtype, int dk, int dv, int64_t lq, int64_t lk, const void* bias) {
  if (dtype != TPA_DTYPE_F32 || dk != dv || (dk != 64 && dk != 128) || bias) return 0;
  // both kernels spend a 128-row block on every head however few rows there are
  if (lq < 64 || lk < 64) return 0;
  return 1;
}

int dense_bwd_f32_launch(const float* q, const float* k, const float* v, const float* d_o, const float* lse, const float* delta,
                         const int32_t* qseg, const int32_t* kvseg, float* dq, float* dk, float* dv, int B, int lq, int lk,
                         int H, int D, float sm_scale, int causal, int coff, hipStream_t stream) {
  tpa::BwdF32Params p{};
  p.q = q; p.k = k; p.v = v; p.d_o = d_o; p.lse = lse; p.delta = delta; p.qseg = qseg; p.kvseg = kvseg;
  p.dq = dq; p.dk = dk; p.dv = dv; p.B = B; p.lq = lq; p.lk = lk; p.H = H; p.sm_scale = sm_scale; p.causal = causal; p.coff = causal ? coff : 0;
  if (qseg) return D == 128 ? tpa::launch_pair<128, true>(p, stream) : tpa::launch_pair<64, true>(p, stream);
  return D == 128 ? tpa::launch_pair<128, false>(p, stream) : tpa::launch_pair<64, false>(p, stream);
}
