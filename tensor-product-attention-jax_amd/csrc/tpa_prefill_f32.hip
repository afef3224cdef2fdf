// Flash-style prefill for fp32 inputs on gfx950: fp32 MFMA contractions, fp32 online softmax.
//
// Same decomposition as the bf16 kernel: one workgroup = one (batch, head, block of 256 query
// rows), eight waves of 32 rows; per tile of 64 keys the workgroup rebuilds the head's K and V
// tile from the rank factors (K = (1/R) sum_r a_r (x) b_r, tpa/tpa.py:364,417) into LDS, as fp32,
// and each wave computes
//     S^T = K Q^T      v_mfma_f32_32x32x2_f32; Q stays in registers, pre-scaled by
//                      sm_scale*log2(e); each lane ends up with 32 logits of ONE query row
//     online softmax   the recurrence of tpa/tpa.py:389-424 with the normalisation deferred
//     O^T += V^T P^T   the S^T accumulator, turned into P in place, is the B operand
// A 32x32x2 step takes two contraction indices, one per half of the wave.  Neither contraction
// cares about the order of its index, so the halves walk it in the order that makes every LDS
// operand read a 16-byte one: over d, half g takes d = 8m + 4g + e (m outer, e = 0..3 from one
// read); over keys, half g takes the key its S^T register already belongs to; and the rows of a
// 32-row block of O^T are d = (D/32) i + block, so one read of V[key][(D/32) i ...] feeds all
// blocks and the epilogue stores whole vectors.
// The matrix pipe is the bound by a wide margin (256 MFMAs of 64 cycles per wave and tile against
// a few hundred vector instructions), so the loop is plain: rebuild the next tile, compute this
// one, one barrier.  The dense baseline (tpa/mha.py:23-37) is the same kernel with rank 1 and
// weight 1.
#include "tpa_common.h"

namespace tpa {
namespace {

constexpr int kTK = 64;   // keys per tile
constexpr int kNW = 8;    // waves per workgroup (32 query rows each); half as many where 256-row blocks are too few

struct F32Params {
  TpaFactor qa, qb, ka, kb, va, vb;  // dense: a pointers null, b = q/k/v with stride_l = H*D
  const int32_t* qseg;
  const int32_t* kvseg;
  const int32_t* kvlen;
  float* o;
  float* lse;
  int B, lq, lk, H, rq, rk;
  float sm_scale;
  int causal, coff, nqb, npairs, groups;  // coff: with causal, row i sees keys <= i + coff; groups: see pair_of_workgroup
};

template <int D>
struct LdsF32 {
  static constexpr int RS = D + 4;        // row stride (floats): 16-byte reads of 16 rows hit distinct banks
  static constexpr int kTile = kTK * RS;  // floats of one tile
  static constexpr size_t kBytes = (size_t)(4 * kTile + 2 * kTK) * 4;  // K and V double buffered + key segment ids
};

template <int D, int NW, bool SEG>
__global__ __launch_bounds__(NW * 64) void prefill_f32_kernel(F32Params pp) {
  constexpr int NT = NW * 64, kBQ = NW * 32;
  constexpr int RS = LdsF32<D>::RS, kTile = LdsF32<D>::kTile;
  constexpr int NDB = D / 32;         // 32-row blocks of O^T
  constexpr int NQ = D / 2;           // Q values per lane
  constexpr int CPR = D / 4;          // 16-byte chunks per row
  constexpr int CH = kTK * CPR / NT;  // chunks per thread, tile and matrix
  static_assert(CH >= 1 && kTK * CPR % NT == 0, "loader shape");
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;

  struct Fac { const float* ptr; int64_t stride_b, stride_l, stride_r; };
  auto fac = [](const TpaFactor& f) { return Fac{static_cast<const float*>(f.ptr), f.stride_b, f.stride_l, f.stride_r}; };
  struct { Fac qa, qb, ka, kb, va, vb; const int32_t* qseg; const int32_t* kvseg; const int32_t* kvlen; float* o; float* lse; int B, lq, lk, H, rq, rk; float sm_scale; int causal, coff, nqb, npairs, groups; } const p = {
      fac(pp.qa), fac(pp.qb), fac(pp.ka), fac(pp.kb), fac(pp.va), fac(pp.vb), pp.qseg, pp.kvseg, pp.kvlen, pp.o, pp.lse,
      pp.B, pp.lq, pp.lk, pp.H, pp.rq, pp.rk, pp.sm_scale, pp.causal, pp.causal ? pp.coff : 0, pp.nqb, pp.npairs, pp.groups};

  extern __shared__ __attribute__((aligned(16))) float smem_f32[];
  float* const lds_k = smem_f32;                                         // [2][kTK][RS]
  float* const lds_v = smem_f32 + 2 * kTile;                             // [2][kTK][RS]
  int32_t* const lds_seg = reinterpret_cast<int32_t*>(smem_f32 + 4 * kTile);  // [2][kTK]

  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;  // heaviest causal blocks first
  const int qblk = p.nqb - 1 - pair / p.B;
  const int b = pair % p.B;

  const int tid = threadIdx.x;
  const int w = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int q0 = qblk * kBQ;
  const int wrow0 = q0 + 32 * w;
  const int qrow = wrow0 + i;
  const int qrow_ld = min(qrow, p.lq - 1);
  const bool dense = p.ka.ptr == nullptr;  // dense q, k, v: weight 1, the head's slice of the row

  // ---- key range
  const int len_b = p.kvlen ? max(0, min(p.kvlen[b], p.lk)) : p.lk;
  const int coff = p.coff + (p.causal == TPA_CAUSAL_BOTTOM_RIGHT ? len_b - p.lq : 0);  // bottom-right alignment counts from the end of this entry's keys
  int kend = p.causal ? min(len_b, min(q0 + kBQ, p.lq) + coff) : len_b, kbeg = 0;
  if constexpr (SEG) {  // only tiles that hold keys with ids of these rows
    if (kend > 0) {
      int first, last;
      id_window<NT>(p.qseg + (int64_t)b * p.lq + q0, min(kBQ, p.lq - q0), p.kvseg + (int64_t)b * p.lk, kend, reinterpret_cast<int32_t*>(smem_f32), tid, first, last);
      kbeg = last < 0 ? 0 : first / kTK * kTK;
      kend = last + 1;
    }
  }
  float* const orow = p.o + (((int64_t)b * p.lq + qrow) * p.H + h) * D;
  if (kend <= 0) {  // no key at all: the rows end as NaN / -inf (tpa/tpa.py:437-439)
    if (qrow < p.lq) {
      const f32x4 nan4 = {__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
#pragma unroll
      for (int cch = 0; cch < D / 8; ++cch) *reinterpret_cast<f32x4*>(orow + 8 * cch + 4 * g) = nan4;
      if (p.lse && g == 0) p.lse[((int64_t)b * p.H + h) * p.lq + qrow] = -INFINITY;
    }
    return;
  }
  const int ntiles = (kend - kbeg + kTK - 1) / kTK;
  const int wave_last_tile = p.causal ? min(ntiles - 1, max(wrow0 + coff + 31 - kbeg, 0) / kTK) : ntiles - 1;

  // ---- Q (B operand of S^T = K Q^T), scaled: qf[4m + e] = c * Q[qrow][8m + 4g + e]
  float qf[NQ];
#pragma unroll
  for (int j = 0; j < NQ; ++j) qf[j] = 0.f;
  {
    const float* qb = p.qb.ptr + b * p.qb.stride_b + (int64_t)qrow_ld * p.qb.stride_l + (dense ? (int64_t)h * D : 0) + 4 * g;
    const float* qa = dense ? nullptr : p.qa.ptr + b * p.qa.stride_b + (int64_t)qrow_ld * p.qa.stride_l + h;
    for (int r = 0; r < p.rq; ++r) {
      const float a = dense ? 1.f : qa[r * p.qa.stride_r];
#pragma unroll
      for (int m = 0; m < D / 8; ++m) {
        const f32x4 bv = *reinterpret_cast<const f32x4*>(qb + r * p.qb.stride_r + 8 * m);
#pragma unroll
        for (int e = 0; e < 4; ++e) qf[4 * m + e] += a * bv[e];
      }
    }
    const float scale = p.sm_scale * kLog2e / (float)p.rq;
#pragma unroll
    for (int j = 0; j < NQ; ++j) qf[j] *= scale;
  }

  // ---- tile rebuild: thread -> CH chunks of 4 floats per matrix
  const float* const kb_b = p.kb.ptr + b * p.kb.stride_b + (dense ? (int64_t)h * D : 0);
  const float* const vb_b = p.vb.ptr + b * p.vb.stride_b + (dense ? (int64_t)h * D : 0);
  const float* const ka_b = dense ? nullptr : p.ka.ptr + b * p.ka.stride_b + h;
  const float* const va_b = dense ? nullptr : p.va.ptr + b * p.va.stride_b + h;
  const float inv_r = 1.f / (float)p.rk;
  auto rebuild = [&](int tile) __attribute__((always_inline)) {
    float* const kd = lds_k + (tile & 1) * kTile;
    float* const vd = lds_v + (tile & 1) * kTile;
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int chunk = q * NT + tid, t = chunk / CPR, cc = chunk % CPR;
      const int tok = kbeg + tile * kTK + t;
      f32x4 ak = {0.f, 0.f, 0.f, 0.f}, av = {0.f, 0.f, 0.f, 0.f};
      if (tok < kend) {  // rows past the end stay zero: they are masked, and 0 * padding must not make NaN
        for (int r = 0; r < p.rk; ++r) {
          const float wk = dense ? 1.f : ka_b[(int64_t)tok * p.ka.stride_l + r * p.ka.stride_r];
          const float wv = dense ? 1.f : va_b[(int64_t)tok * p.va.stride_l + r * p.va.stride_r];
          const f32x4 bk = *reinterpret_cast<const f32x4*>(kb_b + (int64_t)tok * p.kb.stride_l + r * p.kb.stride_r + 4 * cc);
          const f32x4 bv = *reinterpret_cast<const f32x4*>(vb_b + (int64_t)tok * p.vb.stride_l + r * p.vb.stride_r + 4 * cc);
          ak += wk * bk;
          av += wv * bv;
        }
      }
      *reinterpret_cast<f32x4*>(kd + t * RS + 4 * cc) = ak * inv_r;
      *reinterpret_cast<f32x4*>(vd + t * RS + 4 * cc) = av * inv_r;
    }
    if constexpr (SEG)
      if (tid < kTK) lds_seg[(tile & 1) * kTK + tid] = p.kvseg[(int64_t)b * p.lk + min(kbeg + tile * kTK + tid, p.lk - 1)];
  };

  // ---- per-wave state
  f32x16 o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[db][v] = 0.f;
  float m_run = -INFINITY;  // running max of row qrow (log2 domain, scale included)
  float lsum = 0.f;         // this lane's share of sum exp2(x - m_run)
  int32_t qseg = 0;
  if constexpr (SEG) qseg = p.qseg[(int64_t)b * p.lq + qrow_ld];

  f32x16 s[2];  // logits, then probabilities, of the tile in flight: two 32-key blocks
  auto logits_softmax = [&](int tile) __attribute__((always_inline)) {
    const float* const ks = lds_k + (tile & 1) * kTile;
    const int k0 = kbeg + tile * kTK;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int v = 0; v < 16; ++v) s[mb][v] = 0.f;
    // the two blocks' accumulation chains alternate, so no MFMA waits for the one just issued
#pragma unroll
    for (int m = 0; m < D / 8; ++m) {
      const f32x4 kf0 = *reinterpret_cast<const f32x4*>(ks + i * RS + 8 * m + 4 * g);
      const f32x4 kf1 = *reinterpret_cast<const f32x4*>(ks + (32 + i) * RS + 8 * m + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf0[e], qf[4 * m + e], s[0], 0, 0, 0);
        s[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf1[e], qf[4 * m + e], s[1], 0, 0, 0);
      }
    }
    // register v of block mb, wave half g  <->  key k0 + 32 mb + 8 (v / 4) + 4 g + v % 4
    const bool need_mask = (k0 + kTK > kend) || (p.causal && (k0 + kTK - 1 > wrow0 + coff));
    if (need_mask) {
      const int limit = p.causal ? min(qrow + coff, kend - 1) : kend - 1;  // largest visible key index
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int t = k0 + 32 * mb + 8 * (v >> 2) + 4 * g + (v & 3);
          if (t > limit) s[mb][v] = -INFINITY;
        }
    }
    if constexpr (SEG) {  // keys of another segment (tpa/tpa.py:369-375)
      const int32_t* idslot = lds_seg + (tile & 1) * kTK;
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          const int4 ids = *reinterpret_cast<const int4*>(idslot + 32 * mb + 8 * vq + 4 * g);
          if (ids.x != qseg) s[mb][4 * vq] = -INFINITY;
          if (ids.y != qseg) s[mb][4 * vq + 1] = -INFINITY;
          if (ids.z != qseg) s[mb][4 * vq + 2] = -INFINITY;
          if (ids.w != qseg) s[mb][4 * vq + 3] = -INFINITY;
        }
    }
    float tmax = s[0][0];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int v = 0; v < 16; ++v) tmax = fmaxf(tmax, s[mb][v]);
    tmax = halves_max(tmax);
    const float m_new = fmaxf(m_run, tmax);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a row that has met no visible key yet
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);  // 0 while m_run is -inf (nothing accumulated)
    m_run = m_new;
    if (__any(alpha != 1.f)) {
      lsum *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[db][v] *= alpha;
    }
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float pv = __builtin_amdgcn_exp2f(s[mb][v] - m_use);
        lsum += pv;
        s[mb][v] = pv;
      }
  };
  // O^T += V^T P^T: the step of register v takes, in wave half g, the key that register belongs to
  auto accumulate = [&](int tile) __attribute__((always_inline)) {
    const float* const vs = lds_v + (tile & 1) * kTile;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int kr = 32 * mb + 8 * (v >> 2) + 4 * g + (v & 3);
        const f32xN vf = *reinterpret_cast<const f32xN*>(vs + kr * RS + NDB * i);
#pragma unroll
        for (int db = 0; db < NDB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[db], s[mb][v], o[db], 0, 0, 0);
      }
  };

  rebuild(0);
  __syncthreads();
  // The next tile may be rebuilt anywhere between two barriers.  Waves w and w + 4 share a SIMD:
  // one of them rebuilds (waiting for its factor loads) before its matrix work, the other in the
  // middle of it, so the SIMD always has a wave with matrix work and both end the tile together.
  const bool rebuild_first = w < NW / 2;
  for (int j = 0; j < ntiles; ++j) {
    const bool more = j + 1 < ntiles, mine = j <= wave_last_tile && wrow0 < p.lq;  // waves past the last row only help rebuild
    if (rebuild_first && more) rebuild(j + 1);
    if (mine) logits_softmax(j);
    if (!rebuild_first && more) rebuild(j + 1);
    if (mine) accumulate(j);
    __syncthreads();
  }

  // ---- epilogue: row 8 (v / 4) + 4 g + v % 4 of block db is d = NDB * row + db
  const float ltot = halves_sum(lsum);
  const float inv = 1.f / ltot;  // no visible key: 0 * inf = NaN, as in tpa/tpa.py:437-439
  if (qrow < p.lq) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = 8 * (v >> 2) + 4 * g + (v & 3);
      f32xN out;
#pragma unroll
      for (int db = 0; db < NDB; ++db) out[db] = o[db][v] * inv;
      *reinterpret_cast<f32xN*>(orow + NDB * row) = out;
    }
    if (p.lse && g == 0) p.lse[((int64_t)b * p.H + h) * p.lq + qrow] = (m_run + __builtin_amdgcn_logf(ltot)) * kLn2;
  }
}

// ---------------------------------------------------------------------------------------------
// The same for problems with few blocks of 256 query rows.  Such a launch leaves most of the chip idle and its time is
// that of one workgroup walking all keys (one sequence of 512 tokens, 8 heads of 64: 16 workgroups, 75 us).  Here a
// workgroup owns 32 query rows and its NW waves split the keys: wave w takes the tiles of 32 keys w, w + NW, ...,
// rebuilds each into LDS of its own (no barrier in the loop) with the next tile's factors on their way while the matrix
// pipe works on this one, and the partial results are merged through LDS with the rule of _lse_accum
// (tpa/tpa.py:228-242).  Every workgroup rebuilds its tiles for 32 rows instead of 256, which is why the kernel above
// stays the one for launches that fill the chip (`rows_per_workgroup` below).
template <int D, int NW>
struct SplitLdsF32 {
  static constexpr int RS = D + 4;
  static constexpr int kPerWave = 2 * 32 * RS;  // K and V tile; the merge reuses the K tile (O), its last columns (m, l)
  static constexpr size_t kBytes = (size_t)(NW * kPerWave + 4) * 4;
};

template <int D, int NW, bool SEG>
__global__ __launch_bounds__(NW * 64, 1) void prefill_f32_split_kernel(F32Params p) {
  constexpr int RS = SplitLdsF32<D, NW>::RS;
  constexpr int NDB = D / 32, CPR = D / 4, RPI = 64 / CPR, NST = 32 / RPI;  // a load instruction of the wave takes RPI rows
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;

  extern __shared__ __attribute__((aligned(16))) float smem_f32_split[];
  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int qblk = p.nqb - 1 - pair / p.B;  // heaviest causal blocks first
  const int b = pair % p.B;

  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int q0 = qblk * 32, qrow = q0 + i, qrow_ld = min(qrow, p.lq - 1);
  const bool dense = p.ka.ptr == nullptr;  // dense q, k, v: weight 1, the head's slice of the row
  float* const lds_k = smem_f32_split + w * SplitLdsF32<D, NW>::kPerWave;  // [32][RS]
  float* const lds_v = lds_k + 32 * RS;

  const int len_b = p.kvlen ? max(0, min(p.kvlen[b], p.lk)) : p.lk;
  const int coff = !p.causal ? 0 : p.coff + (p.causal == TPA_CAUSAL_BOTTOM_RIGHT ? len_b - p.lq : 0);
  int kend = p.causal ? min(len_b, min(q0 + 32, p.lq) + coff) : len_b, kbeg = 0;
  int32_t qseg = 0;
  if constexpr (SEG) {
    qseg = p.qseg[(int64_t)b * p.lq + qrow_ld];
    if (kend > 0) {
      int first, last;
      id_window<NW * 64>(p.qseg + (int64_t)b * p.lq + q0, min(32, p.lq - q0), p.kvseg + (int64_t)b * p.lk, kend,
                                  reinterpret_cast<int32_t*>(smem_f32_split), tid, first, last);
      kbeg = last < 0 ? 0 : first / 32 * 32;
      kend = last < 0 ? 0 : last + 1;
    }
  }
  const int ntiles = kend > kbeg ? (kend - kbeg + 31) / 32 : 0;

  // Factor rows as raw buffer loads: per array one lane offset that never changes and a scalar one per load (with 64-bit
  // addresses per lane and load the kernel spilled 240 registers).  Tokens from kend on are inside the array or read as
  // zero; the last tile clears them (padding rows may hold anything, and 0 * NaN must not reach the sums).
  const float inv_r = 1.f / (float)p.rk;
  const int lrow = l / CPR, lc = l % CPR;
  struct Rows { __amdgpu_buffer_rsrc_t rs; int voff, sl, sr; };  // byte offset of the lane, bytes between tokens and ranks
  auto rows_of = [&](const TpaFactor& f, int64_t first, int lane_elem, int width) {
    const float* base = static_cast<const float*>(f.ptr) + b * f.stride_b + first;
    const int64_t bytes = ((int64_t)(p.lk - 1) * f.stride_l + (int64_t)(p.rk - 1) * f.stride_r + width) * 4;
    return Rows{__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, (int)bytes, 0x00020000),
                (int)((lrow * f.stride_l + lane_elem) * 4), (int)(f.stride_l * 4), (int)(f.stride_r * 4)};
  };
  const Rows kb_r = rows_of(p.kb, dense ? (int64_t)h * D : 0, 4 * lc, D), vb_r = rows_of(p.vb, dense ? (int64_t)h * D : 0, 4 * lc, D);
  const Rows ka_r = dense ? kb_r : rows_of(p.ka, h, 0, 1), va_r = dense ? vb_r : rows_of(p.va, h, 0, 1);
  struct Flight { f32x4 x[NST]; float wt[NST]; };  // rows in flight and their weights (K's or V's, one rank)
  Flight in;
  f32x4 vac[NST];  // the sum over V's ranks
  int32_t seg_in = 0, seg_id = 0;  // ids of key (this lane's i) of the next tile and of this one
  auto issue_to = [&](Flight& in, const Rows& rb, const Rows& ra, int tile, int r) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      const int t = kbeg + tile * 32 + q * RPI;
      in.x[q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rb.rs, rb.voff, t * rb.sl + r * rb.sr, 0));
      in.wt[q] = 1.f;
      if (!dense) in.wt[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra.rs, ra.voff, t * ra.sl + r * ra.sr, 0));
    }
  };
  auto issue = [&](const Rows& rb, const Rows& ra, int tile, int r) __attribute__((always_inline)) { issue_to(in, rb, ra, tile, r); };
  auto row_of = [&](const Flight& in, int tile, int q) __attribute__((always_inline)) -> f32x4 {
    const f32x4 x = in.wt[q] * inv_r * in.x[q];
    return q * RPI + lrow < kend - kbeg - tile * 32 ? x : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  // K is added up in its LDS tile (free once the logits are done), V in registers until its tile has been used
  auto take_k_of = [&](const Flight& in, int tile, bool first) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      f32x4* const at = reinterpret_cast<f32x4*>(lds_k + (q * RPI + lrow) * RS + 4 * lc);
      const f32x4 x = row_of(in, tile, q);
      *at = first ? x : *at + x;
    }
  };
  auto take_k = [&](int tile, bool first) __attribute__((always_inline)) { take_k_of(in, tile, first); };
  auto take_v = [&](int tile, bool first) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      const f32x4 x = row_of(in, tile, q);
      vac[q] = first ? x : vac[q] + x;
    }
  };
  auto store_v = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NST; ++q) *reinterpret_cast<f32x4*>(lds_v + (q * RPI + lrow) * RS + 4 * lc) = vac[q];
  };
  // all ranks but the last of one array: the first is on its way already, the last one is when this returns
  auto ranks = [&](const Rows& rb, const Rows& ra, int tile, auto&& take) __attribute__((always_inline)) {
    take(tile, true);
    for (int r = 1; r + 1 < p.rk; ++r) {
      issue(rb, ra, tile, r);
      take(tile, false);
    }
    if (p.rk > 1) issue(rb, ra, tile, p.rk - 1);
  };

  Flight in_k;  // of the first tile only: its first ranks of V and of K travel together, ahead of Q's
  if (w < ntiles) {
    issue(vb_r, va_r, w, 0);
    issue_to(in_k, kb_r, ka_r, w, 0);
  }
  // ---- Q, scaled, through LDS (the waves' tiles are not in use yet): the 32 rows are the same for all waves, and read in the
  // layout of the operand every load of every wave would touch 32 cache lines
  for (int idx = tid; idx < 32 * CPR; idx += NW * 64) {
    const int row = idx / CPR, cc = idx % CPR, row_ld = min(q0 + row, p.lq - 1);
    const float* qb = static_cast<const float*>(p.qb.ptr) + b * p.qb.stride_b + (int64_t)row_ld * p.qb.stride_l + (dense ? (int64_t)h * D : 0) + 4 * cc;
    const float* qa = dense ? nullptr : static_cast<const float*>(p.qa.ptr) + b * p.qa.stride_b + (int64_t)row_ld * p.qa.stride_l + h;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    constexpr int G = 6;  // ranks whose loads are in flight together
    for (int r0 = 0; r0 < p.rq; r0 += G) {
      f32x4 bv[G];
      float a[G];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int r = min(r0 + u, p.rq - 1);
        a[u] = dense ? 1.f : qa[r * p.qa.stride_r];
        bv[u] = *reinterpret_cast<const f32x4*>(qb + r * p.qb.stride_r);
      }
#pragma unroll
      for (int u = 0; u < G; ++u)
        if (r0 + u < p.rq) acc += a[u] * bv[u];
    }
    *reinterpret_cast<f32x4*>(smem_f32_split + row * RS + 4 * cc) = acc * (p.sm_scale * kLog2e / (float)p.rq);
  }
  __syncthreads();
  // B operand of S^T = K Q^T: qf[4m + e] = Q[qrow][8m + 4g + e]
  float qf[D / 2];
#pragma unroll
  for (int m = 0; m < D / 8; ++m) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(smem_f32_split + i * RS + 8 * m + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) qf[4 * m + e] = x[e];
  }
  __syncthreads();

  f32x16 o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[db][v] = 0.f;
  float m_run = -INFINITY, lsum = 0.f;

  if (w < ntiles) {
    ranks(vb_r, va_r, w, take_v);
    take_k_of(in_k, w, true);
    for (int r = 1; r < p.rk; ++r) {
      issue_to(in_k, kb_r, ka_r, w, r);
      if (r == 1) {
        take_v(w, false);
        store_v();
      }
      take_k_of(in_k, w, false);
    }
    if (p.rk == 1) store_v();
    if constexpr (SEG) seg_id = p.kvseg[(int64_t)b * p.lk + min(kbeg + w * 32 + i, p.lk - 1)];
  }
  for (int tile = w; tile < ntiles; tile += NW) {
    const int next = tile + NW;
    const bool more = next < ntiles;
    if (more) issue(vb_r, va_r, next, 0);
    f32x16 s, s2;  // two accumulation chains, added at the end
#pragma unroll
    for (int v = 0; v < 16; ++v) { s[v] = 0.f; s2[v] = 0.f; }
#pragma unroll
    for (int m = 0; m < D / 8; ++m) {
      if (m == D / 16 && more) ranks(vb_r, va_r, next, take_v);
      const f32x4 kf = *reinterpret_cast<const f32x4*>(lds_k + i * RS + 8 * m + 4 * g);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[0], qf[4 * m], s, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[1], qf[4 * m + 1], s2, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[2], qf[4 * m + 2], s, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[3], qf[4 * m + 3], s2, 0, 0, 0);
    }
    if (more) {
      if (p.rk > 1) take_v(next, false);
      issue(kb_r, ka_r, next, 0);
      if constexpr (SEG) seg_in = p.kvseg[(int64_t)b * p.lk + min(kbeg + next * 32 + i, p.lk - 1)];
    }
    // register v, wave half g  <->  key k0 + 8 (v / 4) + 4 g + v % 4
    const int k0 = kbeg + tile * 32;
    const int limit = p.causal ? min(qrow + coff, kend - 1) : kend - 1;  // largest visible key index
    float tmax = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int t = 8 * (v >> 2) + 4 * g + (v & 3);
      bool keep = k0 + t <= limit;
      if constexpr (SEG) {
        const int32_t id_t = __shfl(seg_id, t, 64);  // by every lane, whatever it keeps
        keep = keep && id_t == qseg;
      }
      s[v] = keep ? s[v] + s2[v] : -INFINITY;
      tmax = fmaxf(tmax, s[v]);
    }
    tmax = halves_max(tmax);
    const float m_new = fmaxf(m_run, tmax);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a row that has met no visible key yet
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    if (__any(alpha != 1.f)) {
      lsum *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[db][v] *= alpha;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = __builtin_amdgcn_exp2f(s[v] - m_use);
      lsum += s[v];
    }
    // O^T += V^T P^T: the step of register v takes, in wave half g, the key that register belongs to
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      if (v == 8 && more) ranks(kb_r, ka_r, next, take_k);
      const f32xN vf = *reinterpret_cast<const f32xN*>(lds_v + (8 * (v >> 2) + 4 * g + (v & 3)) * RS + NDB * i);
#pragma unroll
      for (int db = 0; db < NDB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[db], s[v], o[db], 0, 0, 0);
    }
    if (more) {
      if (p.rk > 1) take_k(next, false);
      store_v();
      if constexpr (SEG) seg_id = seg_in;
    }
  }

  // ---- merge the waves: row i of a wave's O at lds_k + i RS, its m and l in the four padding columns
  const float ltot = halves_sum(lsum);
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = 8 * (v >> 2) + 4 * g + (v & 3);  // of block db: d = NDB row + db
    f32xN out;
#pragma unroll
    for (int db = 0; db < NDB; ++db) out[db] = o[db][v];
    *reinterpret_cast<f32xN*>(lds_k + i * RS + NDB * row) = out;
  }
  if (g == 0) {
    lds_k[i * RS + D] = m_run;
    lds_k[i * RS + D + 1] = ltot;
  }
  __syncthreads();
  for (int idx = tid; idx < 32 * CPR; idx += NW * 64) {
    const int row = idx / CPR, cc = idx % CPR;
    if (q0 + row >= p.lq) continue;
    const float* const at = smem_f32_split + row * RS;
    float mmax = -INFINITY, lacc = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) mmax = fmaxf(mmax, at[ww * SplitLdsF32<D, NW>::kPerWave + D]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
      const float mw = at[ww * SplitLdsF32<D, NW>::kPerWave + D];
      const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - mmax);
      acc += f * *reinterpret_cast<const f32x4*>(at + ww * SplitLdsF32<D, NW>::kPerWave + 4 * cc);
      lacc += f * at[ww * SplitLdsF32<D, NW>::kPerWave + D + 1];
    }
    const float inv = 1.f / lacc;  // no visible key: 0 * inf = NaN, as in tpa/tpa.py:437-439
    *reinterpret_cast<f32x4*>(p.o + (((int64_t)b * p.lq + q0 + row) * p.H + h) * D + 4 * cc) = acc * inv;
    if (p.lse && cc == 0) p.lse[((int64_t)b * p.H + h) * p.lq + q0 + row] = (mmax + __builtin_amdgcn_logf(lacc)) * kLn2;
  }
}

// The split kernel's buffer offsets take keys of one batch entry below 2 GiB.
bool split_supported(const F32Params& p) {
  const TpaFactor* fs[4] = {&p.ka, &p.kb, &p.va, &p.vb};
  for (const TpaFactor* f : fs)
    if (f->stride_l < 0 || f->stride_r < 0 || (p.lk * f->stride_l + p.rk * f->stride_r + 256) * 4 >= (int64_t(1) << 31)) return false;
  return true;
}

// Eight waves instead of four where a wave then still has a tile and a half: two per SIMD cover each other's waits (four
// hold 276 registers each, so that only one fits).  At head size 64 only: at 128 the tiles of eight waves exceed the LDS.
// Measured, us, causal, heads of 64: 1 x 400
// tokens, 16 heads 32.1 / 23.9; 1 x 512, 8 heads 32.1 / 23.1; 2 x 1000, 8 heads 69.3 / 51.4 (a quarter of it from Q
// through LDS); 1 x 200, 8 heads 17.6 with four.
bool eight_waves_pay(const F32Params& p) { return p.lk >= 384; }

// Rows of a workgroup: 32 (keys split over its waves), 128 or 256.  A launch of 256-row workgroups that does not fill the
// 256 compute units takes as long as one workgroup; with 128 rows (one wave per SIMD) a tile takes half the time, which
// pays as long as they all fit the chip at once - under the causal mask, whose heaviest workgroup is twice the average,
// up to two rounds.  Measured, us with 256 / 128 / 32 rows: 1 x 512 tokens, 8 heads of 64 causal 75 / 41 / 23; 2 x 1000
// 144 / 69 / 51; not causal 4 x 1000 155 / 113 / 222, 8 x 1000 157 / 191 / 441.  32 causal rows at head size 64 also pay
// for up to four rounds of long sequences, whose heaviest workgroup is twice the average however few there are: 4 x 1000
// 146 / 113 / 102, 1 x 4000 489 with 256 / 294; but 1 x 512, 64 heads 64 / 65, and eight rounds: 8 x 1000 149 / 195.
int rows_per_workgroup(const F32Params& p, int D) {
  auto wgs = [&](int rows) { return (int64_t)((p.lq + rows - 1) / rows) * p.B * p.H; };
  if (wgs(32) <= (D == 64 && p.causal && p.lk >= 768 ? 1024 : 512) && split_supported(p)) return 32;
  return wgs(128) <= 256 || (p.causal && wgs(256) <= 256) ? 128 : 256;
}

template <typename K>
int launch_kernel(K kern, bool (&configured)[kMaxDevices], int rows, int threads, size_t lds, F32Params p, hipStream_t stream) {
  p.nqb = (p.lq + rows - 1) / rows;
  p.npairs = p.nqb * p.B;
  p.groups = head_groups(p.npairs, p.H);
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), lds); rc != TPA_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)workgroups_of(p.npairs, p.H, p.groups)), dim3(threads), lds, stream, p);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

template <int D, bool SEG>
int launch_f32(const F32Params& p, hipStream_t stream) {
  static bool configured[4][kMaxDevices] = {};
  const int rows = rows_per_workgroup(p, D);
  if (rows == 32) {
    if constexpr (D == 64)
      if (eight_waves_pay(p)) return launch_kernel(prefill_f32_split_kernel<D, 8, SEG>, configured[3], 32, 512, SplitLdsF32<D, 8>::kBytes, p, stream);
    return launch_kernel(prefill_f32_split_kernel<D, 4, SEG>, configured[0], 32, 256, SplitLdsF32<D, 4>::kBytes, p, stream);
  }
  if (rows == 128) return launch_kernel(prefill_f32_kernel<D, kNW / 2, SEG>, configured[1], 128, kNW * 32, LdsF32<D>::kBytes, p, stream);
  return launch_kernel(prefill_f32_kernel<D, kNW, SEG>, configured[2], 256, kNW * 64, LdsF32<D>::kBytes, p, stream);
}

int launch_any(const F32Params& p, int d, hipStream_t stream) {
  if (p.kvseg) return d == 128 ? launch_f32<128, true>(p, stream) : launch_f32<64, true>(p, stream);
  return d == 128 ? launch_f32<128, false>(p, stream) : launch_f32<64, false>(p, stream);
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }
bool rows_ok(const TpaFactor& f) {  // rows of 4-float vectors
  return aligned16(f.ptr) && f.stride_b % 4 == 0 && f.stride_l % 4 == 0 && f.stride_r % 4 == 0;
}
}  // namespace
}  // namespace tpa

int tpa_prefill_f32_supported(const TpaFwdArgs* a) {
  if (a->dtype != TPA_DTYPE_F32) return 0;
  if (a->dk != a->dv || (a->dk != 64 && a->dk != 128)) return 0;
  if (!tpa::rows_ok(a->qb) || !tpa::rows_ok(a->kb) || !tpa::rows_ok(a->vb) || !tpa::aligned16(a->o)) return 0;
  return 1;
}

int tpa_prefill_f32_launch(const TpaFwdArgs* a, hipStream_t stream) {
  using namespace tpa;
  F32Params p{};
  p.qa = a->qa; p.qb = a->qb; p.ka = a->ka; p.kb = a->kb; p.va = a->va; p.vb = a->vb;
  p.qseg = a->q_segment_ids; p.kvseg = a->kv_segment_ids; p.kvlen = a->kv_lengths;
  p.o = static_cast<float*>(a->o); p.lse = a->lse;
  p.B = a->B; p.lq = a->lq; p.lk = a->lk; p.H = a->H; p.rq = a->rq; p.rk = a->rk;
  p.sm_scale = a->sm_scale; p.causal = a->causal; p.coff = causal_offset_of(a);
  return launch_any(p, a->dk, stream);
}

int mha_prefill_f32_supported(const MhaFwdArgs* a) {
  if (a->dtype != TPA_DTYPE_F32) return 0;
  if (a->dk != a->dv || (a->dk != 64 && a->dk != 128)) return 0;
  if (a->bias) return 0;
  if (!tpa::aligned16(a->q) || !tpa::aligned16(a->k) || !tpa::aligned16(a->v) || !tpa::aligned16(a->o)) return 0;
  return 1;
}

int mha_prefill_f32_launch(const MhaFwdArgs* a, hipStream_t stream) {
  using namespace tpa;
  F32Params p{};
  const int64_t hd = (int64_t)a->H * a->dk;
  p.qb = TpaFactor{a->q, a->lq * hd, hd, 0};
  p.kb = TpaFactor{a->k, a->lk * hd, hd, 0};
  p.vb = TpaFactor{a->v, a->lk * hd, hd, 0};
  p.qa = p.ka = p.va = TpaFactor{nullptr, 0, 0, 0};
  p.o = static_cast<float*>(a->o); p.lse = a->lse;
  p.B = a->B; p.lq = a->lq; p.lk = a->lk; p.H = a->H; p.rq = 1; p.rk = 1;
  p.sm_scale = a->sm_scale; p.causal = a->causal ? TPA_CAUSAL_TOP_LEFT : TPA_CAUSAL_NONE;
  return launch_any(p, a->dk, stream);
}
