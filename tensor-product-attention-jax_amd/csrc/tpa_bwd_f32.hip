// Backward of dense attention in fp32 on gfx950: fp32 MFMA contractions (v_mfma_f32_32x32x2_f32).
//
// Inputs are dense fp32 Q, K, V, dO [B, l, H, D], LSE [B, H, lq] (natural log) and
// delta = rowsum(O * dO) [B, H, lq]; outputs dense fp32 dQ, dK, dV.  With p = exp(x - lse):
//     dV = p^T dO,  dP = dO V^T,  dS = sm_scale * p * (dP - delta),  dQ = dS K,  dK = dS^T Q
// (tpa/tpa.py:546-995 computes the same quantities per block pair).  Two kernels, each of which
// owns its output rows and therefore needs no atomics:
//   bwd_f32_dq_kernel   workgroup = 128 query rows (4 waves x 32) of one head, loops over key tiles
//   bwd_f32_dkv_kernel  workgroup = 128 keys (4 waves x 32) of one head, loops over query tiles
// The operand placement is that of the fp32 forward kernel: the wave's own 32 rows (queries or
// keys) stay in registers as B operands, so a lane holds the logits of ONE of its rows; the
// streamed tile (64 rows, double buffered in LDS) supplies the A operands with 16-byte reads in
// both roles - as rows (contraction over d: wave half g takes d = 8m + 4g + e) and transposed
// (contraction over the tile's rows: half g takes the row its accumulator register belongs to,
// and the 32 output rows of block db are d = (D/32) i + db) - and the p / dS accumulators are used
// in place as the B operands of the second contraction.
// One wave per SIMD (the register budget of 512 is what holds the wave's rows, two accumulators
// and the next tile in flight); the matrix pipe is the bound by a wide margin.
#include "tpa_common.h"

namespace tpa {
namespace {

constexpr int kTile = 64;    // rows of the streamed tile
constexpr int kWaves = 4;    // waves per workgroup
constexpr int kBlock = 128;  // rows a workgroup owns (32 per wave)
constexpr int kThreads = kWaves * 64;

struct BwdF32Params {
  const float *q, *k, *v, *d_o, *lse, *delta;
  const int32_t *qseg, *kvseg;
  float *dq, *dk, *dv;
  int B, lq, lk, H;
  float sm_scale;
  int causal, coff, nblk, npairs, groups;  // coff: with causal, row i sees keys <= i + coff; groups: see pair_of_workgroup
};

template <int D>
struct BwdLds {
  static constexpr int RS = D + 4;          // row stride (floats)
  static constexpr int kMat = kTile * RS;   // floats of one tile of one matrix
  // two matrices double buffered, then per buffer: lse2[64], delta[64], segment ids[64]
  static constexpr size_t kBytes = (size_t)(4 * kMat + 2 * 3 * kTile) * 4;
};

// The 64 x D tile of dense X[b, row0 .., h, :] that `issue` fetched, into LDS; rows >= nrows as zeros.
template <int D>
struct TileRegs {
  static constexpr int CPR = D / 4, CH = kTile * CPR / kThreads;
  f32x4 r[CH];
  __device__ __forceinline__ void issue(const float* base, int64_t row_stride, int row0, int nrows, bool scrub_nan) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int chunk = c * kThreads + threadIdx.x, t = chunk / CPR, cc = chunk % CPR;
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      if (row0 + t < nrows) x = *reinterpret_cast<const f32x4*>(base + (int64_t)(row0 + t) * row_stride + 4 * cc);
      if (scrub_nan) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = x[e] == x[e] ? x[e] : 0.f;
      }
      r[c] = x;
    }
  }
  __device__ __forceinline__ void store(float* dst) const {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int chunk = c * kThreads + threadIdx.x, t = chunk / CPR, cc = chunk % CPR;
      *reinterpret_cast<f32x4*>(dst + t * BwdLds<D>::RS + 4 * cc) = r[c];
    }
  }
};

// the wave's own row (B operand of the row-wise contractions): out[4m + e] = scale * X[row][8m + 4g + e]
template <int D>
__device__ __forceinline__ void load_own_row(const float* rowp, int g, float scale, bool scrub_nan, float (&out)[D / 2]) {
#pragma unroll
  for (int m = 0; m < D / 8; ++m) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(rowp + 8 * m + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float y = x[e];
      if (scrub_nan) y = y == y ? y : 0.f;
      out[4 * m + e] = y * scale;
    }
  }
}

// acc0 / acc1 (rows 0-31 / 32-63 of the tile, lane = own row) = tile rows . own row, over d
template <int D>
__device__ __forceinline__ void rows_dot(const float* tile, int i, int g, const float (&own)[D / 2], f32x16& acc0, f32x16& acc1) {
  constexpr int RS = BwdLds<D>::RS;
#pragma unroll
  for (int v = 0; v < 16; ++v) { acc0[v] = 0.f; acc1[v] = 0.f; }
#pragma unroll
  for (int m = 0; m < D / 8; ++m) {
    const f32x4 a0 = *reinterpret_cast<const f32x4*>(tile + i * RS + 8 * m + 4 * g);
    const f32x4 a1 = *reinterpret_cast<const f32x4*>(tile + (32 + i) * RS + 8 * m + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[e], own[4 * m + e], acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[e], own[4 * m + e], acc1, 0, 0, 0);
    }
  }
}

// out[db] (rows d = (D/32) i + db, lane = own row) += tile^T . w, over the tile's rows; w0 / w1 are
// accumulators of rows_dot's layout (register v, half g <-> tile row 32 mb + 8 (v/4) + 4 g + v%4)
template <int D>
__device__ __forceinline__ void cols_accumulate(const float* tile, int i, int g, const f32x16& w0, const f32x16& w1, f32x16 (&out)[D / 32]) {
  constexpr int RS = BwdLds<D>::RS, NDB = D / 32;
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = 32 * mb + 8 * (v >> 2) + 4 * g + (v & 3);
      const f32xN a = *reinterpret_cast<const f32xN*>(tile + row * RS + NDB * i);
      const float wv = mb == 0 ? w0[v] : w1[v];
#pragma unroll
      for (int db = 0; db < NDB; ++db) out[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[db], wv, out[db], 0, 0, 0);
    }
}

template <int D>
__device__ __forceinline__ void store_own_row(float* rowp, int g, const f32x16 (&acc)[D / 32]) {
  constexpr int NDB = D / 32;
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = 8 * (v >> 2) + 4 * g + (v & 3);
    f32xN out;
#pragma unroll
    for (int db = 0; db < NDB; ++db) out[db] = acc[db][v];
    *reinterpret_cast<f32xN*>(rowp + NDB * row) = out;
  }
}

// ------------------------------------------------------------------------------------- dQ
template <int D, bool SEG>
__global__ __launch_bounds__(kThreads) void bwd_f32_dq_kernel(BwdF32Params p) {
  constexpr int kMat = BwdLds<D>::kMat, NDB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float smem_bwd_f32[];
  float* const lds_k = smem_bwd_f32;             // [2][kTile][RS]
  float* const lds_v = smem_bwd_f32 + 2 * kMat;  // [2][kTile][RS]
  int32_t* const lds_seg = reinterpret_cast<int32_t*>(smem_bwd_f32 + 4 * kMat);  // [2][kTile] key segment ids

  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int blk = p.nblk - 1 - pair / p.B;  // heaviest causal blocks first
  const int b = pair % p.B;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int q0 = blk * kBlock, wrow0 = q0 + 32 * w, qrow = wrow0 + i, qrow_ld = min(qrow, p.lq - 1);
  const int64_t hd = (int64_t)p.H * D;

  int kend = p.causal ? max(1, min(p.lk, q0 + kBlock + p.coff)) : p.lk, kbeg = 0;  // at least one (then fully masked) tile
  if constexpr (SEG) {  // only tiles that hold keys with ids of these rows
    int first, last;
    id_window<kThreads>(p.qseg + (int64_t)b * p.lq + q0, min(kBlock, p.lq - q0), p.kvseg + (int64_t)b * p.lk, kend, reinterpret_cast<int32_t*>(smem_bwd_f32), tid, first, last);
    kbeg = last < 0 ? 0 : first / kTile * kTile;
    kend = last < 0 ? 1 : last + 1;
  }
  const int ntiles = (kend - kbeg + kTile - 1) / kTile;
  const int wave_last_tile = p.causal ? min(ntiles - 1, max(wrow0 + p.coff + 31 - kbeg, 0) / kTile) : ntiles - 1;

  float qf[D / 2], gf[D / 2];
  load_own_row<D>(p.q + ((int64_t)b * p.lq + qrow_ld) * hd + (int64_t)h * D, g, p.sm_scale * kLog2e, false, qf);
  load_own_row<D>(p.d_o + ((int64_t)b * p.lq + qrow_ld) * hd + (int64_t)h * D, g, 1.f, true, gf);
  const float lse = p.lse[((int64_t)b * p.H + h) * p.lq + qrow_ld];
  // a row without a visible key (lse = -inf) has no gradient: +inf makes every p of the row zero
  const float lse2 = (qrow < p.lq && lse > -INFINITY) ? lse * kLog2e : INFINITY;
  const float delta = p.delta[((int64_t)b * p.H + h) * p.lq + qrow_ld];
  int32_t qseg = 0;
  if constexpr (SEG) qseg = p.qseg[(int64_t)b * p.lq + qrow_ld];

  f32x16 dq[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) dq[db][v] = 0.f;

  const float* const kbase = p.k + (int64_t)b * p.lk * hd + (int64_t)h * D;
  const float* const vbase = p.v + (int64_t)b * p.lk * hd + (int64_t)h * D;
  TileRegs<D> kreg, vreg;
  int32_t seg_reg = 0;
  auto issue = [&](int tile) __attribute__((always_inline)) {
    kreg.issue(kbase, hd, kbeg + tile * kTile, kend, false);
    vreg.issue(vbase, hd, kbeg + tile * kTile, kend, false);
    if constexpr (SEG)
      if (tid < kTile) seg_reg = p.kvseg[(int64_t)b * p.lk + min(kbeg + tile * kTile + tid, p.lk - 1)];
  };
  auto commit = [&](int tile) __attribute__((always_inline)) {
    kreg.store(lds_k + (tile & 1) * kMat);
    vreg.store(lds_v + (tile & 1) * kMat);
    if constexpr (SEG)
      if (tid < kTile) lds_seg[(tile & 1) * kTile + tid] = seg_reg;
  };

  auto compute = [&](int tile) __attribute__((always_inline)) {
    const float* const ks = lds_k + (tile & 1) * kMat;
    const float* const vs = lds_v + (tile & 1) * kMat;
    const int k0 = kbeg + tile * kTile;
    f32x16 s[2], dp[2];
    rows_dot<D>(ks, i, g, qf, s[0], s[1]);    // x * log2(e)
    rows_dot<D>(vs, i, g, gf, dp[0], dp[1]);  // dP
    const int limit = p.causal ? min(qrow + p.coff, kend - 1) : kend - 1;  // largest visible key index
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
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
          const float pt = keep ? __builtin_amdgcn_exp2f(s[mb][v] - lse2) : 0.f;
          s[mb][v] = p.sm_scale * pt * (dp[mb][v] - delta);  // dS
        }
      }
    cols_accumulate<D>(ks, i, g, s[0], s[1], dq);
  };

  issue(0);
  commit(0);
  __syncthreads();
  for (int j = 0; j < ntiles; ++j) {
    const bool more = j + 1 < ntiles;
    if (more) issue(j + 1);
    if (j <= wave_last_tile) compute(j);
    if (more) commit(j + 1);
    __syncthreads();
  }
  if (qrow < p.lq) store_own_row<D>(p.dq + ((int64_t)b * p.lq + qrow) * hd + (int64_t)h * D, g, dq);
}

// ------------------------------------------------------------------------------------- dK, dV
template <int D, bool SEG>
__global__ __launch_bounds__(kThreads) void bwd_f32_dkv_kernel(BwdF32Params p) {
  constexpr int kMat = BwdLds<D>::kMat, NDB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float smem_bwd_f32[];
  float* const lds_q = smem_bwd_f32;             // [2][kTile][RS]
  float* const lds_g = smem_bwd_f32 + 2 * kMat;  // [2][kTile][RS]  upstream gradient rows
  float* const lds_row = smem_bwd_f32 + 4 * kMat;  // [2][lse2 | delta | segment id][kTile]

  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int blk = pair / p.B;  // under the causal mask the first key blocks see the most rows: heaviest first
  const int b = pair % p.B;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int k0 = blk * kBlock, wkey0 = k0 + 32 * w, key = wkey0 + i, key_ld = min(key, p.lk - 1);
  const int64_t hd = (int64_t)p.H * D;

  // under the causal mask only rows at or after a key see it
  int first_tile = p.causal ? max(k0 - p.coff, 0) / kTile : 0;
  int ntiles = (p.lq + kTile - 1) / kTile;
  if constexpr (SEG) {  // only tiles that hold rows with ids of these keys
    int first, last;
    const int rbeg = min(first_tile * kTile, p.lq);
    id_window<kThreads>(p.kvseg + (int64_t)b * p.lk + k0, min(kBlock, p.lk - k0), p.qseg + (int64_t)b * p.lq + rbeg, p.lq - rbeg, reinterpret_cast<int32_t*>(smem_bwd_f32), tid, first, last);
    ntiles = last < 0 ? 0 : (rbeg + last) / kTile + 1;
    if (last >= 0) first_tile = (rbeg + first) / kTile;
  }
  const int wave_first_tile = p.causal ? max(wkey0 - p.coff, 0) / kTile : 0;

  float kf[D / 2], vf[D / 2];
  load_own_row<D>(p.k + ((int64_t)b * p.lk + key_ld) * hd + (int64_t)h * D, g, p.sm_scale * kLog2e, false, kf);
  load_own_row<D>(p.v + ((int64_t)b * p.lk + key_ld) * hd + (int64_t)h * D, g, 1.f, false, vf);
  int32_t kseg = 0;
  if constexpr (SEG) kseg = p.kvseg[(int64_t)b * p.lk + key_ld];

  f32x16 dk[NDB], dv[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) { dk[db][v] = 0.f; dv[db][v] = 0.f; }

  const float* const qbase = p.q + (int64_t)b * p.lq * hd + (int64_t)h * D;
  const float* const gbase = p.d_o + (int64_t)b * p.lq * hd + (int64_t)h * D;
  const float* const lse_b = p.lse + ((int64_t)b * p.H + h) * p.lq;
  const float* const delta_b = p.delta + ((int64_t)b * p.H + h) * p.lq;
  TileRegs<D> qreg, greg;
  float row_reg = 0.f;  // threads 0-63: lse2, 64-127: delta, 128-191: segment id of one row of the tile
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
  auto commit = [&](int tile) __attribute__((always_inline)) {
    qreg.store(lds_q + (tile & 1) * kMat);
    greg.store(lds_g + (tile & 1) * kMat);
    if (tid < 3 * kTile) lds_row[(tile & 1) * 3 * kTile + tid] = row_reg;
  };

  auto compute = [&](int tile) __attribute__((always_inline)) {
    const float* const qs = lds_q + (tile & 1) * kMat;
    const float* const gs = lds_g + (tile & 1) * kMat;
    const float* const rows = lds_row + (tile & 1) * 3 * kTile;
    const int r0 = tile * kTile;
    f32x16 s[2], dp[2];
    rows_dot<D>(qs, i, g, kf, s[0], s[1]);    // x * log2(e); lane = key, registers = rows of the tile
    rows_dot<D>(gs, i, g, vf, dp[0], dp[1]);  // dP
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
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
          const float pt = keep ? __builtin_amdgcn_exp2f(s[mb][v] - lse2[e]) : 0.f;
          s[mb][v] = pt;                                            // p
          dp[mb][v] = p.sm_scale * pt * (dp[mb][v] - dl[e]);        // dS
        }
      }
    cols_accumulate<D>(gs, i, g, s[0], s[1], dv);
    cols_accumulate<D>(qs, i, g, dp[0], dp[1], dk);
  };

  if (first_tile < ntiles) {
    issue(first_tile);
    commit(first_tile);
  }
  __syncthreads();
  for (int j = first_tile; j < ntiles; ++j) {
    const bool more = j + 1 < ntiles;
    if (more) issue(j + 1);
    if (j >= wave_first_tile) compute(j);
    if (more) commit(j + 1);
    __syncthreads();
  }
  if (key < p.lk) {
    store_own_row<D>(p.dk + ((int64_t)b * p.lk + key) * hd + (int64_t)h * D, g, dk);
    store_own_row<D>(p.dv + ((int64_t)b * p.lk + key) * hd + (int64_t)h * D, g, dv);
  }
}

// ---------------------------------------------------------------------------------------------
// The same two kernels for problems with few blocks of 128 rows (or keys), whose launch leaves most of the chip idle and
// takes as long as one workgroup walking the whole sequence (2 sequences of 1000 tokens, 8 heads of 64: 128 workgroups,
// 112 and 160 us).  A workgroup owns 32 rows (keys) and its NW waves split the streamed tiles, 32 rows each: wave w
// takes tiles w, w + NW, ... into LDS of its own (no barrier in the loop; the next tile's rows are in flight in registers
// meanwhile, one matrix at a time), and the partial sums are added through LDS in a fixed order.
template <int D>
struct SplitLds {
  static constexpr int RS = D + 4;
  static constexpr int kMat = 32 * RS;
  static constexpr int kPerWave = 2 * kMat + 3 * 32;  // two matrices, then lse2 | delta | segment id of the tile's rows
  static constexpr size_t bytes(int nw) { return (size_t)nw * kPerWave * 4; }
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
  static __device__ __forceinline__ void store(const Regs& r, float* dst, int l, bool scrub_nan) {
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      f32x4 x = r[q];
      if (scrub_nan) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = x[e] == x[e] ? x[e] : 0.f;
      }
      *reinterpret_cast<f32x4*>(dst + (q * RPI + l / CPR) * SplitLds<D>::RS + 4 * (l % CPR)) = x;
    }
  }
};

// a = A-tile rows . own row, b = B-tile rows . own row, both over d: two chains that alternate
template <int D>
__device__ __forceinline__ void rows_dot_pair(const float* ta, const float* tb, int i, int g, const float (&oa)[D / 2], const float (&ob)[D / 2], f32x16& a, f32x16& b) {
  constexpr int RS = SplitLds<D>::RS;
#pragma unroll
  for (int v = 0; v < 16; ++v) { a[v] = 0.f; b[v] = 0.f; }
#pragma unroll
  for (int m = 0; m < D / 8; ++m) {
    const f32x4 fa = *reinterpret_cast<const f32x4*>(ta + i * RS + 8 * m + 4 * g);
    const f32x4 fb = *reinterpret_cast<const f32x4*>(tb + i * RS + 8 * m + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], oa[4 * m + e], a, 0, 0, 0);
      b = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[e], ob[4 * m + e], b, 0, 0, 0);
    }
  }
}

template <int D>
__device__ __forceinline__ void cols_accumulate32(const float* tile, int i, int g, const f32x16& wgt, f32x16 (&out)[D / 32]) {
  constexpr int RS = SplitLds<D>::RS, NDB = D / 32;
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const f32xN a = *reinterpret_cast<const f32xN*>(tile + (8 * (v >> 2) + 4 * g + (v & 3)) * RS + NDB * i);
#pragma unroll
    for (int db = 0; db < NDB; ++db) out[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[db], wgt[v], out[db], 0, 0, 0);
  }
}

// a wave's accumulator as rows of 32 own rows x D in LDS
template <int D>
__device__ __forceinline__ void park(float* dst, int i, int g, const f32x16 (&acc)[D / 32]) { store_own_row<D>(dst + i * SplitLds<D>::RS, g, acc); }

// dst[row0 + r, h, :] = sum over the waves of what they parked at `at`
template <int D, int NW>
__device__ __forceinline__ void add_waves(const float* at, float* dst, int row0, int nrows, int64_t hd, int tid) {
  constexpr int CPR = D / 4;
  for (int idx = tid; idx < 32 * CPR; idx += NW * 64) {
    const int r = idx / CPR, cc = idx % CPR;
    if (row0 + r >= nrows) break;
    f32x4 x = *reinterpret_cast<const f32x4*>(at + r * SplitLds<D>::RS + 4 * cc);
#pragma unroll
    for (int w = 1; w < NW; ++w) x += *reinterpret_cast<const f32x4*>(at + w * SplitLds<D>::kPerWave + r * SplitLds<D>::RS + 4 * cc);
    *reinterpret_cast<f32x4*>(dst + (int64_t)(row0 + r) * hd + 4 * cc) = x;
  }
}

template <int D, int NW, bool SEG>
__global__ __launch_bounds__(NW * 64, 1) void bwd_f32_dq_split_kernel(BwdF32Params p) {
  constexpr int NDB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float smem_bwd_f32[];
  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int blk = p.nblk - 1 - pair / p.B, b = pair % p.B;  // heaviest causal blocks first
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
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
  if (w < ntiles) vt.issue(kbeg + 32 * w, in);

  float qf[D / 2], gf[D / 2];
  load_own_row<D>(p.q + ((int64_t)b * p.lq + qrow_ld) * hd + (int64_t)h * D, g, p.sm_scale * kLog2e, false, qf);
  load_own_row<D>(p.d_o + ((int64_t)b * p.lq + qrow_ld) * hd + (int64_t)h * D, g, 1.f, true, gf);
  const float lse = p.lse[((int64_t)b * p.H + h) * p.lq + qrow_ld];
  // a row without a visible key (lse = -inf) has no gradient: +inf makes every p of the row zero
  const float lse2 = (qrow < p.lq && lse > -INFINITY) ? lse * kLog2e : INFINITY;
  const float delta = p.delta[((int64_t)b * p.H + h) * p.lq + qrow_ld];
  f32x16 dq[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) dq[db][v] = 0.f;

  auto next_k = [&](int tile) __attribute__((always_inline)) {
    WaveTile<D>::store(in, lds_v, l, false);
    kt.issue(kbeg + 32 * tile, in);
    if constexpr (SEG) seg_in = p.kvseg[(int64_t)b * p.lk + min(kbeg + 32 * tile + i, p.lk - 1)];
  };
  auto arrive_k = [&]() __attribute__((always_inline)) {
    WaveTile<D>::store(in, lds_k, l, false);
    if constexpr (SEG) lds_seg[i] = seg_in;
  };
  if (w < ntiles) {
    next_k(w);
    arrive_k();
  }
  for (int tile = w; tile < ntiles; tile += NW) {
    const bool more = tile + NW < ntiles;
    if (more) vt.issue(kbeg + 32 * (tile + NW), in);
    const int k0 = kbeg + 32 * tile;
    f32x16 s, dp;
    rows_dot_pair<D>(lds_k, lds_v, i, g, qf, gf, s, dp);
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
    cols_accumulate32<D>(lds_k, i, g, s, dq);
    if (more) arrive_k();
  }
  park<D>(lds_k, i, g, dq);
  __syncthreads();
  add_waves<D, NW>(smem_bwd_f32, p.dq + (int64_t)b * p.lq * hd + (int64_t)h * D, q0, p.lq, hd, tid);
}

template <int D, int NW, bool SEG>
__global__ __launch_bounds__(NW * 64, 1) void bwd_f32_dkv_split_kernel(BwdF32Params p) {
  constexpr int NDB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float smem_bwd_f32[];
  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int blk = pair / p.B, b = pair % p.B;  // under the causal mask the first key blocks see the most rows: heaviest first
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
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
  if (w < ntiles) gt.issue(rbeg + 32 * w, in);
  auto next_q = [&](int tile) __attribute__((always_inline)) {
    const int row0 = rbeg + 32 * tile, r = row0 + i;
    WaveTile<D>::store(in, lds_g, l, true);
    qt.issue(row0, in);
    const float x = (g ? delta_b : lse_b)[min(r, p.lq - 1)];
    // rows past the end and rows without a visible key (lse = -inf): +inf makes every p of the row zero
    row_in = g ? x : (r < rend && x > -INFINITY) ? x * kLog2e : INFINITY;
    if constexpr (SEG) seg_in = p.qseg[(int64_t)b * p.lq + min(r, p.lq - 1)];
  };
  auto arrive_q = [&]() __attribute__((always_inline)) {
    WaveTile<D>::store(in, lds_q, l, false);
    lds_row[l] = row_in;
    if constexpr (SEG) reinterpret_cast<int32_t*>(lds_row)[64 + i] = seg_in;
  };

  float kf[D / 2], vf[D / 2];
  load_own_row<D>(p.k + ((int64_t)b * p.lk + key_ld) * hd + (int64_t)h * D, g, p.sm_scale * kLog2e, false, kf);
  load_own_row<D>(p.v + ((int64_t)b * p.lk + key_ld) * hd + (int64_t)h * D, g, 1.f, false, vf);
  f32x16 dk[NDB], dv[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) { dk[db][v] = 0.f; dv[db][v] = 0.f; }

  if (w < ntiles) {
    next_q(w);
    arrive_q();
  }
  for (int tile = w; tile < ntiles; tile += NW) {
    const bool more = tile + NW < ntiles;
    if (more) gt.issue(rbeg + 32 * (tile + NW), in);
    const int r0 = rbeg + 32 * tile;
    f32x16 s, dp;
    rows_dot_pair<D>(lds_q, lds_g, i, g, kf, vf, s, dp);  // lane = key, registers = rows of the tile
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
    cols_accumulate32<D>(lds_g, i, g, s, dv);
    if (more) next_q(tile + NW);
    cols_accumulate32<D>(lds_q, i, g, dp, dk);
    if (more) arrive_q();
  }
  park<D>(lds_q, i, g, dk);
  park<D>(lds_g, i, g, dv);
  __syncthreads();
  add_waves<D, NW>(smem_bwd_f32, p.dk + (int64_t)b * p.lk * hd + (int64_t)h * D, k0, p.lk, hd, tid);
  add_waves<D, NW>(smem_bwd_f32 + SplitLds<D>::kMat, p.dv + (int64_t)b * p.lk * hd + (int64_t)h * D, k0, p.lk, hd, tid);
}

// Whether 32-row workgroups pay: the launch of 128-row ones leaves half of the 256 compute units idle, or fills them once
// with causal blocks, of which the heaviest is twice the average.  (Forward and backward, us, 128 / 32 rows, 8 heads of
// 64: 2 x 1000 tokens causal 384 / 215, not causal 434 / 313; 4 x 1000 causal 461 / 387, not causal 470 / 511; 8 x 1000
// causal 562 / 617.)  The split kernels' buffer offsets take a batch entry below 2 GiB.
bool few_blocks(const BwdF32Params& p, int rows, int D) {
  const int64_t big = p.lq > p.lk ? p.lq : p.lk;
  return (int64_t)((rows + kBlock - 1) / kBlock) * p.B * p.H <= (p.causal ? 256 : 128) && (big + 64) * p.H * D * 4 < (int64_t(1) << 31);
}

// Eight waves instead of four, as in the forward (tpa_prefill_f32.hip): head size 64, a tile and a half per wave.  Forward
// and backward, us, causal, 8 heads of 64: 1 x 400 tokens 93 -> 81, 2 x 1000 198 -> 167, 2 x 2000 622 -> 500.
template <int D>
bool eight_waves_pay(int streamed) { return D == 64 && streamed >= 384; }

template <typename K>
int launch_kernel(K kern, bool (&configured)[kMaxDevices], int rows, int block, int threads, size_t lds, BwdF32Params p, hipStream_t stream) {
  p.nblk = (rows + block - 1) / block;
  p.npairs = p.nblk * p.B;
  p.groups = head_groups(p.npairs, p.H);
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), lds); rc != TPA_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)workgroups_of(p.npairs, p.H, p.groups)), dim3(threads), lds, stream, p);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

template <int D, bool SEG>
int launch_pair(const BwdF32Params& p, hipStream_t stream) {
  static bool configured[6][kMaxDevices] = {};
  auto dq = [&]() {
    if (!few_blocks(p, p.lq, D)) return launch_kernel(bwd_f32_dq_kernel<D, SEG>, configured[1], p.lq, kBlock, kThreads, BwdLds<D>::kBytes, p, stream);
    if constexpr (D == 64)
      if (eight_waves_pay<D>(p.lk)) return launch_kernel(bwd_f32_dq_split_kernel<D, 8, SEG>, configured[4], p.lq, 32, 512, SplitLds<D>::bytes(8), p, stream);
    return launch_kernel(bwd_f32_dq_split_kernel<D, 4, SEG>, configured[0], p.lq, 32, 256, SplitLds<D>::bytes(4), p, stream);
  };
  auto dkv = [&]() {
    if (!few_blocks(p, p.lk, D)) return launch_kernel(bwd_f32_dkv_kernel<D, SEG>, configured[3], p.lk, kBlock, kThreads, BwdLds<D>::kBytes, p, stream);
    if constexpr (D == 64)
      if (eight_waves_pay<D>(p.lq)) return launch_kernel(bwd_f32_dkv_split_kernel<D, 8, SEG>, configured[5], p.lk, 32, 512, SplitLds<D>::bytes(8), p, stream);
    return launch_kernel(bwd_f32_dkv_split_kernel<D, 4, SEG>, configured[2], p.lk, 32, 256, SplitLds<D>::bytes(4), p, stream);
  };
  if (int rc = dq(); rc != TPA_OK) return rc;
  return dkv();
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
