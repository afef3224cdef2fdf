// Flash-style prefill for fp32 inputs on gfx950: fp32 contractions as split bf16 products, fp32 online softmax.
//
// Same decomposition as the bf16 kernel: one workgroup = one (batch, head, block of 256 query
// rows), eight waves of 32 rows; per tile of keys the workgroup rebuilds the head's K and V
// tile from the rank factors (K = (1/R) sum_r a_r (x) b_r, tpa/tpa.py:364,417) in fp32, splits every
// value into three bf16 parts (tpa_split3.h) and stages them as three planes in LDS; each wave computes
//     S^T = K Q^T      six v_mfma_f32_32x32x16_bf16 per 16 values of d; Q stays in registers, pre-scaled by
//                      sm_scale*log2(e) and split; each lane ends up with the logits of ONE query row
//     online softmax   the recurrence of tpa/tpa.py:389-424 with the normalisation deferred
//     O^T += V^T P^T   P is split in the registers of the logits it was made from
// The contraction over keys does not care about their order, so the B operand of a step of 16 keys is the accumulator
// as it is - half g of the wave holds keys 8q + 4g + 0..3 of two neighbouring q - and V is read transposed to match.
// The fp32 matrix instruction, which this kernel used to be made of, takes 64 cycles for 2 contraction indices where the
// six of a split take 192 for 16: 4 x 4096 tokens, 16 heads of 128 causal 2497 -> 1593 us (174 TFLOP/s where the fp32
// instruction peaks at 157), 2 x 2000, 64 heads of 64 712 -> 487.  It is left for workgroups that meet values that do not
// split (tpa_split3.h): these walk their tiles a second time.
// The loop is plain: rebuild the next tile, compute this one, one barrier.  The dense baseline (tpa/mha.py:23-37) is the
// same kernel with rank 1 and weight 1.
#include <algorithm>
#include <type_traits>

#include "tpa_common.h"
#include "tpa_split3.h"

namespace tpa {
namespace {

constexpr int kNW = 8;    // waves per workgroup (32 query rows each); half as many where 256-row blocks are too few

struct F32Params {
  TpaFactor qa, qb, ka, kb, va, vb;  // dense: a pointers null, b = q/k/v with stride_l = H*D
  const int32_t* qseg;
  const int32_t* kvseg;
  const int32_t* kvlen;
  float* o;
  float* lse;
  int B, lq, lk, H, rq, rk;
  float q_scale;  // of the sum over Q's ranks: sm_scale log2(e) / rq, or 1 for a dense Q that has it already
  int causal, coff, nqb, npairs, groups;  // coff: with causal, row i sees keys <= i + coff; groups: see pair_of_workgroup
};

template <int D>
struct LdsF32 {
  static constexpr int kTK = D == 128 ? 32 : 64;  // keys per tile: two buffers of six planes fit the LDS
  static constexpr int KS = D + 8, VS = D + 32;   // row strides (bf16): spread the banks for the row reads of K and the transposed ones of V
  static constexpr int kKPlane = kTK * KS, kVPlane = kTK * VS;
  static constexpr int kBuffer = 3 * (kKPlane + kVPlane);  // bf16 elements of one buffer
  static constexpr size_t kBytes = (size_t)2 * kBuffer * 2 + 2 * kTK * 4;  // two buffers, key segment ids
};

template <int D, int NW, bool SEG>
__global__ __launch_bounds__(NW * 64) void prefill_f32_kernel(F32Params pp) {
  constexpr int NT = NW * 64, kBQ = NW * 32;
  typedef LdsF32<D> L;
  constexpr int kTK = L::kTK, NMB = kTK / 32;  // keys of a tile, 32-key blocks
  constexpr int NDB = D / 32;         // 32-row blocks of O^T
  constexpr int NKS = D / 16;         // steps of the contraction over d
  constexpr int CPR = D / 4;          // 16-byte chunks per row
  constexpr int CH = kTK * CPR / NT;  // chunks per thread, tile and matrix
  static_assert(CH >= 1 && kTK * CPR % NT == 0, "loader shape");

  struct Fac { const float* ptr; int64_t stride_b, stride_l, stride_r; };
  auto fac = [](const TpaFactor& f) { return Fac{static_cast<const float*>(f.ptr), f.stride_b, f.stride_l, f.stride_r}; };
  struct { Fac qa, qb, ka, kb, va, vb; const int32_t* qseg; const int32_t* kvseg; const int32_t* kvlen; float* o; float* lse; int B, lq, lk, H, rq, rk; float q_scale; int causal, coff, nqb, npairs, groups; } const p = {
      fac(pp.qa), fac(pp.qb), fac(pp.ka), fac(pp.kb), fac(pp.va), fac(pp.vb), pp.qseg, pp.kvseg, pp.kvlen, pp.o, pp.lse,
      pp.B, pp.lq, pp.lk, pp.H, pp.rq, pp.rk, pp.q_scale, pp.causal, pp.causal ? pp.coff : 0, pp.nqb, pp.npairs, pp.groups};

  extern __shared__ __attribute__((aligned(16))) float smem_f32[];
  uint16_t* const planes = reinterpret_cast<uint16_t*>(smem_f32);  // [2][K h, m, l; V h, m, l]
  int32_t* const lds_seg = reinterpret_cast<int32_t*>(planes + 2 * L::kBuffer);  // [2][kTK]

  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;  // heaviest causal blocks first
  const int qblk = p.nqb - 1 - pair / p.B;
  const int b = pair % p.B;

  const int tid = threadIdx.x;
  const int w = scalar(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
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

  // ---- Q (B operand of S^T = K Q^T), scaled and split: lane (i, g) holds Q[qrow][16 ks + 8 g + 0..7].  `fp32` is a compile-time
  // flag here and below: the walk over the tiles that uses the fp32 instruction
  Split3 qf[NKS];
  bool bad = false;  // this thread has met values that do not split
  auto load_q = [&](auto fp32) __attribute__((always_inline)) {
    const float* const qb = p.qb.ptr + b * p.qb.stride_b + (int64_t)qrow_ld * p.qb.stride_l + (dense ? (int64_t)h * D : 0) + 8 * g;
    const float* const qa = dense ? nullptr : p.qa.ptr + b * p.qa.stride_b + (int64_t)qrow_ld * p.qa.stride_l + h;
    const float scale = p.q_scale;
    float top = 0.f;
    constexpr int NH = NKS < 4 ? NKS : 4;  // steps at a time
#pragma unroll
    for (int k0 = 0; k0 < NKS; k0 += NH) {
      float q[NH][8];
#pragma unroll
      for (int ks = 0; ks < NH; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) q[ks][e] = 0.f;
      for (int r = 0; r < p.rq; ++r) {
        const float a = dense ? 1.f : qa[r * p.qa.stride_r];
#pragma unroll
        for (int j = 0; j < 2 * NH; ++j) {
          const f32x4 bv = *reinterpret_cast<const f32x4*>(qb + r * p.qb.stride_r + 16 * (k0 + (j >> 1)) + 4 * (j & 1));
#pragma unroll
          for (int e = 0; e < 4; ++e) q[j >> 1][4 * (j & 1) + e] += a * bv[e];
        }
      }
#pragma unroll
      for (int ks = 0; ks < NH; ++ks) {
#pragma unroll
        for (int e = 0; e < 8; ++e) q[ks][e] *= scale;
#pragma unroll
        for (int e = 0; e < 8; e += 2) top = largest(top, q[ks][e], q[ks][e + 1]);
        qf[k0 + ks] = split8<decltype(fp32)::value>(q[ks]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    bad |= !(top < kLogitOperand);
  };

  // ---- tile rebuild: thread -> CH chunks of 4 floats per matrix
  const float* const kb_b = p.kb.ptr + b * p.kb.stride_b + (dense ? (int64_t)h * D : 0);
  const float* const vb_b = p.vb.ptr + b * p.vb.stride_b + (dense ? (int64_t)h * D : 0);
  const float* const ka_b = dense ? nullptr : p.ka.ptr + b * p.ka.stride_b + h;
  const float* const va_b = dense ? nullptr : p.va.ptr + b * p.va.stride_b + h;
  const float inv_r = 1.f / (float)p.rk;
  auto stage = [&](auto fp32, uint16_t* at, int plane, const f32x4& x) __attribute__((always_inline)) {
    constexpr bool whole = decltype(fp32)::value;
    const Pair3 a = whole ? halves_of_pair(x[0], x[1]) : split_pair(x[0], x[1]), c = whole ? halves_of_pair(x[2], x[3]) : split_pair(x[2], x[3]);
    *reinterpret_cast<u32x2*>(at) = u32x2{a.h, c.h};
    *reinterpret_cast<u32x2*>(at + plane) = u32x2{a.m, c.m};
    if constexpr (!whole) *reinterpret_cast<u32x2*>(at + 2 * plane) = u32x2{a.l, c.l};
  };
  auto rebuild = [&](auto fp32, int tile) __attribute__((always_inline)) {
    uint16_t* const kd = planes + (tile & 1) * L::kBuffer;
    uint16_t* const vd = kd + 3 * L::kKPlane;
    float k_top = 0.f;
    Magnitudes v_seen;
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
      ak *= inv_r;
      av *= inv_r;
      k_top = largest(k_top, ak);
      v_seen.add(av);
      stage(fp32, kd + t * L::KS + 4 * cc, L::kKPlane, ak);
      stage(fp32, vd + t * L::VS + 4 * cc, L::kVPlane, av);
    }
    if constexpr (!decltype(fp32)::value) bad |= !(k_top < kLogitOperand) | v_seen.irregular();
    if constexpr (SEG)
      if (tid < kTK) lds_seg[(tile & 1) * kTK + tid] = p.kvseg[(int64_t)b * p.lk + min(kbeg + tile * kTK + tid, p.lk - 1)];
  };
  auto row_operand = [&](const uint16_t* at) __attribute__((always_inline)) -> Split3 {  // eight values of a row of K
    return {*reinterpret_cast<const bf16x8*>(at), *reinterpret_cast<const bf16x8*>(at + L::kKPlane), *reinterpret_cast<const bf16x8*>(at + 2 * L::kKPlane)};
  };

  // ---- per-wave state
  f32x16 o[NDB];
  float m_run, lsum;  // running max of row qrow (log2 domain, scale included); this lane's share of sum exp2(x - m_run)
  int32_t qseg = 0;
  if constexpr (SEG) qseg = p.qseg[(int64_t)b * p.lq + qrow_ld];
  const TileIds<SEG, 1> ids_of_wave({qseg});

  f32x16 s[NMB];  // logits, then probabilities, of the tile in flight
  auto logits_softmax = [&](auto fp32, int tile) __attribute__((always_inline)) {
    const uint16_t* const kt = planes + (tile & 1) * L::kBuffer + i * L::KS + 8 * g;
    const int k0 = kbeg + tile * kTK;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
      for (int v = 0; v < 16; ++v) s[mb][v] = 0.f;
    if constexpr (!decltype(fp32)::value) {
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        f32x16 small;
#pragma unroll
        for (int v = 0; v < 16; ++v) small[v] = 0.f;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          const Split3 kf = row_operand(kt + 32 * mb * L::KS + 16 * ks);
          mfma_small(kf, qf[ks], small);
          s[mb] = mfma_bf16(kf.h, qf[ks].h, s[mb]);
          if constexpr (D == 128) __builtin_amdgcn_sched_barrier(0);  // the operands of one step at a time: more do not fit the registers
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) s[mb][v] += small[v];
        bad |= too_large(s[mb]);  // -inf + inf is NaN where the fp32 instruction has -inf: the key drops out
      }
    } else {
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) mfma_joined(row_operand(kt + 32 * mb * L::KS + 16 * ks), qf[ks], s[mb]);
    }
    // register v of block mb, wave half g  <->  key k0 + 32 mb + 8 (v / 4) + 4 g + v % 4
    const bool need_mask = (k0 + kTK > kend) || (p.causal && (k0 + kTK - 1 > wrow0 + coff));
    if (need_mask) {
      const int limit = p.causal ? min(qrow + coff, kend - 1) : kend - 1;  // largest visible key index
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int t = k0 + 32 * mb + 8 * (v >> 2) + 4 * g + (v & 3);
          if (t > limit) s[mb][v] = -INFINITY;
        }
    }
    if constexpr (SEG) {  // keys of another segment (tpa/tpa.py:369-375)
      const int32_t* idslot = lds_seg + (tile & 1) * kTK;
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb)
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
    for (int mb = 0; mb < NMB; ++mb)
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
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float pv = __builtin_amdgcn_exp2f(s[mb][v] - m_use);
        lsum += pv;
        s[mb][v] = pv;
      }
  };
  // O^T += V^T P^T, 16 keys at a time: registers 8t .. 8t + 7 of a block are keys 8 (2t + u) + 4 g + 0..3 for u = 0, 1
  const int lp = l & 15, dhalf = (l >> 4) & 1;
  auto accumulate = [&](auto fp32, int tile) __attribute__((always_inline)) {
    const uint16_t* const vt = planes + (tile & 1) * L::kBuffer + 3 * L::kKPlane + (4 * g + (lp >> 2)) * L::VS + 16 * dhalf + 4 * (lp & 3);
    auto column_operand = [&](int mb, int t, int db) __attribute__((always_inline)) -> Split3 {
      bf16x8 part[3];
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) {
        const uint16_t* const at = vt + pl * L::kVPlane + (32 * mb + 16 * t) * L::VS + 32 * db;
        const s16x4 u0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)at);
        const s16x4 u1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(at + 8 * L::VS));
        part[pl] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(u0, u1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
      return {part[0], part[1], part[2]};
    };
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = s[mb][8 * t + e];
        if constexpr (!decltype(fp32)::value) {
          const Split3 pf = split8(x);
#pragma unroll
          for (int db = 0; db < NDB; db += 2) {  // the accumulation chains of two blocks alternate
            const Split3 v0 = column_operand(mb, t, db), v1 = column_operand(mb, t, db + 1);
            o[db] = mfma_bf16(v0.l, pf.h, o[db]);
            o[db + 1] = mfma_bf16(v1.l, pf.h, o[db + 1]);
            o[db] = mfma_bf16(v0.h, pf.l, o[db]);
            o[db + 1] = mfma_bf16(v1.h, pf.l, o[db + 1]);
            o[db] = mfma_bf16(v0.m, pf.m, o[db]);
            o[db + 1] = mfma_bf16(v1.m, pf.m, o[db + 1]);
            o[db] = mfma_bf16(v0.m, pf.h, o[db]);
            o[db + 1] = mfma_bf16(v1.m, pf.h, o[db + 1]);
            o[db] = mfma_bf16(v0.h, pf.m, o[db]);
            o[db + 1] = mfma_bf16(v1.h, pf.m, o[db + 1]);
            o[db] = mfma_bf16(v0.h, pf.h, o[db]);
            o[db + 1] = mfma_bf16(v1.h, pf.h, o[db + 1]);
            if constexpr (D == 128) __builtin_amdgcn_sched_barrier(0);
          }
        } else {
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            const Split3 vf = column_operand(mb, t, db);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(join(vf, e), x[e], o[db], 0, 0, 0);
          }
        }
      }
  };

  auto walk = [&](auto fp32) __attribute__((always_inline)) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[db][v] = 0.f;
    m_run = -INFINITY;
    lsum = 0.f;
    load_q(fp32);
    rebuild(fp32, 0);
    __syncthreads();
    // The next tile may be rebuilt anywhere between two barriers.  Waves w and w + 4 share a SIMD:
    // one of them rebuilds (waiting for its factor loads) before its matrix work, the other in the
    // middle of it, so the SIMD always has a wave with matrix work and both end the tile together.
    const bool rebuild_first = w < NW / 2;
    for (int j = 0; j < ntiles; ++j) {
      const bool more = j + 1 < ntiles;
      const bool mine = j <= wave_last_tile && wrow0 < p.lq &&  // waves past the last row, or whose documents a tile has not, only help rebuild
                        ids_of_wave.look(lds_seg + (j & 1) * kTK, l & (kTK - 1)) != kNoneOfThem;
      if (rebuild_first && more) rebuild(fp32, j + 1);
      if (mine) logits_softmax(fp32, j);
      if (!rebuild_first && more) rebuild(fp32, j + 1);
      if (mine) accumulate(fp32, j);
      __syncthreads();
    }
  };
  walk(std::false_type{});
  if (__builtin_expect(__syncthreads_or(bad), 0)) walk(std::true_type{});

  // ---- epilogue: register v of block db is d = 32 db + 8 (v / 4) + 4 g + v % 4
  const float ltot = halves_sum(lsum);
  const float inv = 1.f / ltot;  // no visible key: 0 * inf = NaN, as in tpa/tpa.py:437-439
  if (qrow < p.lq) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        f32x4 out;
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = o[db][4 * vq + e] * inv;
        *reinterpret_cast<f32x4*>(orow + 32 * db + 8 * vq + 4 * g) = out;
      }
    if (p.lse && g == 0) p.lse[((int64_t)b * p.H + h) * p.lq + qrow] = (m_run + __builtin_amdgcn_logf(ltot)) * kLn2;
  }
}

// ---------------------------------------------------------------------------------------------
// The same for problems with few blocks of 256 query rows.  Such a launch leaves most of the chip idle and its time is
// that of one workgroup walking all keys (one sequence of 512 tokens, 8 heads of 64: 16 workgroups, 53 us).  Here a
// workgroup owns 32 query rows and its NW waves split the keys: wave w takes the tiles of 32 keys w, w + NW, ...,
// rebuilds each into LDS of its own (no barrier in the loop; fp32, split on the way to the matrix cores: a value has one
// reader) with the next tile's factors on their way while they work on this one, and the partial results are merged
// through LDS with the rule of _lse_accum (tpa/tpa.py:228-242).  One workgroup's chain of loads, rebuild and two
// contractions is the bound: 1 x 512 tokens, 8 heads of 64 causal 23.4 us with the fp32 instruction and offsets that the
// compiler did not know to be scalar (a loop around every load), 17.1 so; 2 x 1000 51 -> 37.  Every workgroup rebuilds its tiles for 32 rows instead of 256, which is why the kernel above
// stays the one for launches that fill the chip (`rows_per_workgroup` below).
template <int D>
struct SplitLdsF32 {
  // waves: two per SIMD cover each other's waits (four or eight, us, heads of 64: 1 x 128 tokens, 8 heads 9.6 / 8.6, 1 x 384
  // 18.3 / 13.9, 4 x 448 27.5 / 22.5); at head size 128 the tiles of eight exceed the LDS
  static constexpr int NW = D == 64 ? 8 : 4;
  static constexpr int RS = D + 4;
  static constexpr int kPerWave = 2 * 32 * RS;  // K and V tile; the merge reuses the K tile (O), its last columns (m, l)
  static constexpr int QS = D + 8;              // row stride (bf16) of the parts of Q, which all waves read
  static constexpr int kQPlane = 32 * QS;
  static constexpr size_t kBytes = (size_t)NW * kPerWave * 4 + (size_t)3 * kQPlane * 2;
};

template <int D, bool SEG, int RK>  // RK: rank of K and V, 0 = any
__global__ __launch_bounds__(SplitLdsF32<D>::NW * 64, 1) void prefill_f32_split_kernel(F32Params p) {
  constexpr int RS = SplitLdsF32<D>::RS, NW = SplitLdsF32<D>::NW;
  constexpr int NDB = D / 32, CPR = D / 4, RPI = 64 / CPR, NST = 32 / RPI;  // a load instruction of the wave takes RPI rows
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;

  extern __shared__ __attribute__((aligned(16))) float smem_f32_split[];
  int pair, h;
  if (!pair_of_workgroup(blockIdx.x, p.npairs, p.H, p.B, p.groups, pair, h)) return;
  const int qblk = p.nqb - 1 - pair / p.B;  // heaviest causal blocks first
  const int b = pair % p.B;

  // the wave's index is a scalar: the scalar offsets of its buffer loads are made from it
  const int tid = threadIdx.x, w = scalar(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
  const int q0 = qblk * 32, qrow = q0 + i, qrow_ld = min(qrow, p.lq - 1);
  const int rk = RK ? RK : p.rk;
  const bool dense = RK == 1 && p.ka.ptr == nullptr;  // dense q, k, v: weight 1, the head's slice of the row
  float* const lds_k = smem_f32_split + w * SplitLdsF32<D>::kPerWave;  // [32][RS]
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
  kbeg = __builtin_amdgcn_readfirstlane(kbeg);
  kend = __builtin_amdgcn_readfirstlane(kend);
  const int ntiles = kend > kbeg ? (kend - kbeg + 31) / 32 : 0;

  // Factor rows as raw buffer loads: per array one lane offset that never changes and a scalar one per load (with 64-bit
  // addresses per lane and load the kernel spilled 240 registers).  Tokens from kend on are inside the array or read as
  // zero; the last tile clears them (padding rows may hold anything, and 0 * NaN must not reach the sums).
  const float inv_r = 1.f / (float)rk;
  const int lrow = l / CPR, lc = l % CPR;
  struct Rows { __amdgpu_buffer_rsrc_t rs; int voff, sl, sr; };  // byte offset of the lane, bytes between tokens and ranks
  auto rows_of = [&](const TpaFactor& f, int64_t first, int lane_elem, int width) {
    const float* base = static_cast<const float*>(f.ptr) + b * f.stride_b + first;
    const int64_t bytes = ((int64_t)(p.lk - 1) * f.stride_l + (int64_t)(rk - 1) * f.stride_r + width) * 4;
    return Rows{__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, (int)bytes, 0x00020000),
                (int)((lrow * f.stride_l + lane_elem) * 4), (int)(f.stride_l * 4), (int)(f.stride_r * 4)};
  };
  const Rows kb_r = rows_of(p.kb, dense ? (int64_t)h * D : 0, 4 * lc, D), vb_r = rows_of(p.vb, dense ? (int64_t)h * D : 0, 4 * lc, D);
  const Rows ka_r = dense ? kb_r : rows_of(p.ka, h, 0, 1), va_r = dense ? vb_r : rows_of(p.va, h, 0, 1);
  struct Flight { f32x4 x[NST]; float wt[NST]; };  // rows in flight and their weights (K's or V's, one rank)
  f32x4 vac[NST];  // the sum over V's ranks
  int32_t seg_in = 0, seg_id = 0;  // ids of key (this lane's i) of the next tile and of this one
  auto issue = [&](Flight& in, const Rows& rb, const Rows& ra, int tile, int r) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      const int t = kbeg + tile * 32 + q * RPI;
      in.x[q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rb.rs, rb.voff, t * rb.sl + r * rb.sr, 0));
    }
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      const int t = kbeg + tile * 32 + q * RPI;
      in.wt[q] = dense ? 1.f : __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra.rs, ra.voff, t * ra.sl + r * ra.sr, 0));
    }
  };
  auto row_of = [&](const Flight& in, int tile, int q) __attribute__((always_inline)) -> f32x4 {
    const f32x4 x = in.wt[q] * inv_r * in.x[q];
    return q * RPI + lrow < kend - kbeg - tile * 32 ? x : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  // K is added up in its LDS tile (free once the logits are done), V in registers until its tile has been used
  auto take_k = [&](const Flight& in, int tile, bool first) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      f32x4* const at = reinterpret_cast<f32x4*>(lds_k + (q * RPI + lrow) * RS + 4 * lc);
      const f32x4 x = row_of(in, tile, q);
      *at = first ? x : *at + x;
    }
  };
  auto take_v = [&](const Flight& in, int tile, bool first) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      const f32x4 x = row_of(in, tile, q);
      vac[q] = first ? x : vac[q] + x;
    }
  };
  // all ranks but the last of one array: the first is on its way already, the last one is when this returns
  auto but_last = [&](Flight& in, const Rows& rb, const Rows& ra, int tile, auto&& take) __attribute__((always_inline)) {
    if (rk == 1) return;
    take(in, tile, true);
    issue(in, rb, ra, tile, 1);
    for (int r = 2; r < rk; ++r) {
      take(in, tile, false);
      issue(in, rb, ra, tile, r);
    }
  };
  // the last ones; `bad`: this lane has met values that do not split
  bool bad = false;
  auto store_v = [&]() __attribute__((always_inline)) {
    float top = 0.f, bottom = INFINITY;
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      top = largest(top, vac[q]);
      bottom = smallest(bottom, vac[q]);
      *reinterpret_cast<f32x4*>(lds_v + (q * RPI + lrow) * RS + 4 * lc) = vac[q];
    }
    bad |= !(top < 0x1p127f);
    if (bottom < 0x1p-90f) {  // zeros or small values
      Magnitudes seen;
#pragma unroll
      for (int q = 0; q < NST; ++q) seen.add(vac[q]);
      bad |= seen.irregular();
    }
  };
  auto last_k = [&](const Flight& in, int tile) __attribute__((always_inline)) {
    float top = 0.f;
    auto finish = [&](bool first) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < NST; ++q) {
        f32x4* const at = reinterpret_cast<f32x4*>(lds_k + (q * RPI + lrow) * RS + 4 * lc);
        f32x4 x = row_of(in, tile, q);
        if (!first) x += *at;
        top = largest(top, x);
        *at = x;
      }
    };
    if (rk == 1) finish(true);
    else finish(false);
    bad |= !(top < kLogitOperand);
  };

  // At any rank V and K take turns with one set of registers: the last rank of V is waited for before the first of K is requested.
  // (With a set for each up to 317 registers were spilled: 2 x 1000 tokens, 8 heads, rank 4, causal, D = 64 57.6 / 51.8 us, D = 128
  // 150 / 133, with documents of 150 tokens 87 / 77.)
  constexpr bool kTurns = RK == 0;
  Flight in_v, in_k_own;
  Flight& in_k = kTurns ? in_v : in_k_own;
  auto take_last_v = [&](int tile) __attribute__((always_inline)) {
    if (rk == 1) take_v(in_v, tile, true);
    else take_v(in_v, tile, false);
  };
  auto request_first = [&]() __attribute__((always_inline)) {
    if (w < ntiles) {
      issue(in_v, vb_r, va_r, w, 0);
      if constexpr (!kTurns) issue(in_k, kb_r, ka_r, w, 0);
    }
  };
  request_first();  // ahead of Q
  // ---- Q, scaled and split (B operand of S^T = K Q^T): the 32 rows are the same for all waves, which read them from LDS
  uint16_t* const lds_q = reinterpret_cast<uint16_t*>(smem_f32_split + NW * SplitLdsF32<D>::kPerWave);
  auto park_q = [&](auto fp32, const auto& p, int tid) __attribute__((always_inline)) {
    constexpr bool whole = decltype(fp32)::value;
    float top = 0.f;
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
      acc *= p.q_scale;
      top = largest(top, acc);
      const Pair3 x = whole ? halves_of_pair(acc[0], acc[1]) : split_pair(acc[0], acc[1]), y = whole ? halves_of_pair(acc[2], acc[3]) : split_pair(acc[2], acc[3]);
      uint16_t* const at = lds_q + row * SplitLdsF32<D>::QS + 4 * cc;
      *reinterpret_cast<u32x2*>(at) = u32x2{x.h, y.h};
      *reinterpret_cast<u32x2*>(at + SplitLdsF32<D>::kQPlane) = u32x2{x.m, y.m};
      *reinterpret_cast<u32x2*>(at + 2 * SplitLdsF32<D>::kQPlane) = u32x2{x.l, y.l};
    }
    bad |= !(top < kLogitOperand);
    __syncthreads();
  };
  park_q(std::false_type{}, p, tid);
  int q_offset = i * SplitLdsF32<D>::QS + 8 * g;
  auto q_operand = [&](int ks) __attribute__((always_inline)) -> Split3 {
    const uint16_t* const at = lds_q + q_offset + 16 * ks;
    return {*reinterpret_cast<const bf16x8*>(at), *reinterpret_cast<const bf16x8*>(at + SplitLdsF32<D>::kQPlane),
            *reinterpret_cast<const bf16x8*>(at + 2 * SplitLdsF32<D>::kQPlane)};
  };

  f32x16 o[NDB];
  float m_run, lsum;
  auto walk = [&](auto fp32) __attribute__((always_inline)) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[db][v] = 0.f;
    m_run = -INFINITY;
    lsum = 0.f;
    if (w < ntiles) {
      but_last(in_v, vb_r, va_r, w, take_v);
      if constexpr (kTurns) {
        take_last_v(w);
        issue(in_k, kb_r, ka_r, w, 0);
      }
      but_last(in_k, kb_r, ka_r, w, take_k);
      if constexpr (!kTurns) take_last_v(w);
      store_v();
      last_k(in_k, w);
      if constexpr (SEG) seg_id = p.kvseg[(int64_t)b * p.lk + min(kbeg + w * 32 + i, p.lk - 1)];
    }
    for (int tile = w; tile < ntiles; tile += NW) {
      const int next = tile + NW;
      const bool more = next < ntiles, ahead = more && !decltype(fp32)::value;  // the second walk fetches a tile when it is needed: it holds less
      if (ahead) issue(in_v, vb_r, va_r, next, 0);
      f32x16 s;
#pragma unroll
      for (int v = 0; v < 16; ++v) s[v] = 0.f;
      asm volatile("" : "+v"(q_offset));  // Q is read again for every tile: held in registers it would not fit
      if constexpr (!decltype(fp32)::value) {
        f32x16 s2;
#pragma unroll
        for (int v = 0; v < 16; ++v) s2[v] = 0.f;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) {
          float x[8];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const f32x4 kf = *reinterpret_cast<const f32x4*>(lds_k + i * RS + 16 * ks + 8 * g + 4 * u);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[4 * u + e] = kf[e];
          }
          const Split3 kf = split8(x), qf = q_operand(ks);
          mfma_small(kf, qf, s2);
          s = mfma_bf16(kf.h, qf.h, s);
          __builtin_amdgcn_sched_barrier(0);  // the operands of one step at a time: more do not fit the registers
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] += s2[v];
        bad |= too_large(s);  // -inf + inf is NaN where the fp32 instruction has -inf: the key drops out
      } else {
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) {
          const Split3 qf = q_operand(ks);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(lds_k[i * RS + 16 * ks + 8 * g + e], join(qf, e), s, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (ahead) {
        but_last(in_v, vb_r, va_r, next, take_v);
        if constexpr (kTurns) take_last_v(next);
        issue(in_k, kb_r, ka_r, next, 0);
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
        s[v] = keep ? s[v] : -INFINITY;
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
      // O^T += V^T P^T: 16 keys a step, in wave half g those its registers 8t .. 8t + 7 belong to
      auto v_rows = [&](int v) __attribute__((always_inline)) -> f32xN {
        return *reinterpret_cast<const f32xN*>(lds_v + (8 * (v >> 2) + 4 * g + (v & 3)) * RS + NDB * i);
      };
      if constexpr (!decltype(fp32)::value) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if (t == 1 && ahead) but_last(in_k, kb_r, ka_r, next, take_k);
          float x[8], y[NDB][8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            x[e] = s[8 * t + e];
            const f32xN vf = v_rows(8 * t + e);
#pragma unroll
            for (int db = 0; db < NDB; ++db) y[db][e] = vf[db];
          }
          const Split3 pf = split8(x);
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            const Split3 vf = split8(y[db]);
            mfma_small(vf, pf, o[db]);
            o[db] = mfma_bf16(vf.h, pf.h, o[db]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const f32xN vf = v_rows(v);
#pragma unroll
          for (int db = 0; db < NDB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[db], s[v], o[db], 0, 0, 0);
        }
      }
      if (more && !ahead) {
        issue(in_v, vb_r, va_r, next, 0);
        but_last(in_v, vb_r, va_r, next, take_v);
        if constexpr (kTurns) take_last_v(next);
        issue(in_k, kb_r, ka_r, next, 0);
        but_last(in_k, kb_r, ka_r, next, take_k);
        if constexpr (SEG) seg_in = p.kvseg[(int64_t)b * p.lk + min(kbeg + next * 32 + i, p.lk - 1)];
      }
      if (more) {
        if constexpr (!kTurns) take_last_v(next);
        store_v();
        last_k(in_k, next);
        if constexpr (SEG) seg_id = seg_in;
      }
    }
    // ---- for the merge of the waves: row i of a wave's O at lds_k + i RS, its m and l in the four padding columns
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
  };
  walk(std::false_type{});
  if (__builtin_expect(__syncthreads_or(bad), 0)) {
    request_first();
    park_q(std::true_type{}, *arguments_again<F32Params>(), again(tid));
    walk(std::true_type{});
    __syncthreads();
  }
  // ---- merge the waves
  for (int idx = tid; idx < 32 * CPR; idx += NW * 64) {
    const int row = idx / CPR, cc = idx % CPR;
    if (q0 + row >= p.lq) continue;
    const float* const at = smem_f32_split + row * RS;
    float mmax = -INFINITY, lacc = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) mmax = fmaxf(mmax, at[ww * SplitLdsF32<D>::kPerWave + D]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
      const float mw = at[ww * SplitLdsF32<D>::kPerWave + D];
      const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - mmax);
      acc += f * *reinterpret_cast<const f32x4*>(at + ww * SplitLdsF32<D>::kPerWave + 4 * cc);
      lacc += f * at[ww * SplitLdsF32<D>::kPerWave + D + 1];
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

// Rows of a workgroup: 32 (keys split over its waves), 128 or 256.  A launch of 256-row workgroups that does not fill the
// 256 compute units takes as long as one workgroup walking all keys.  Measured, us with 256 / 128 / 32 rows:
//   two rounds of 32-row workgroups at most: 1 x 512 tokens, 8 heads of 64 causal 53 / 52 / 17, 2 x 1000 95 / 97 / 38, not
//   causal 100 / 98 / 57; 2 x 512, 16 heads of 128 causal 109 / 105 / 60
//   up to four under the causal mask, whose heaviest workgroup is twice the average: 8 heads of 64, 8 x 512 56 / 55 / 51,
//   4 x 1000 97 / 97 / 70, 1 x 4000 360 / 429 / 200, but eight rounds 8 x 1000 103 / 118 / 138; with heads of 128 only long
//   sequences: 16 heads, 1 x 2000 360 / 422 / 332, 2 x 1000 188 / 209 / 188, 4 x 512 111 / 108 / 115
//   short sequences whose 128-row workgroups fit the chip at once: 16 heads of 128, 8 x 256 71 / 66 / 78, 4 x 512 not
//   causal 115 / 110 / 170, but 1 x 2000 371 / 435
int rows_per_workgroup(const F32Params& p, int D) {
  auto wgs = [&](int rows) { return (int64_t)((p.lq + rows - 1) / rows) * p.B * p.H; };
  if (wgs(32) <= (p.causal && (D == 64 || p.lk >= 1536) ? 1024 : 512) && split_supported(p)) return 32;
  return wgs(128) <= 256 && p.lk <= (p.causal ? 512 : 1024) ? 128 : 256;
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

template <int D, bool SEG, int RK>
int launch_split(const F32Params& p, hipStream_t stream) {
  static bool configured[kMaxDevices] = {};
  constexpr int NW = SplitLdsF32<D>::NW;
  return launch_kernel(prefill_f32_split_kernel<D, SEG, RK>, configured, 32, NW * 64, SplitLdsF32<D>::kBytes, p, stream);
}

template <int D, bool SEG>
int launch_f32(const F32Params& p, hipStream_t stream) {
  static bool configured[2][kMaxDevices] = {};
  const int rows = rows_per_workgroup(p, D);
  if (rows == 32) {
    if (p.rk == 1) return launch_split<D, SEG, 1>(p, stream);
    return p.rk == 2 ? launch_split<D, SEG, 2>(p, stream) : launch_split<D, SEG, 0>(p, stream);
  }
  if (rows == 128) return launch_kernel(prefill_f32_kernel<D, kNW / 2, SEG>, configured[0], 128, kNW * 32, LdsF32<D>::kBytes, p, stream);
  return launch_kernel(prefill_f32_kernel<D, kNW, SEG>, configured[1], 256, kNW * 64, LdsF32<D>::kBytes, p, stream);
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

namespace tpa {
namespace {
int64_t dense_slot(int64_t floats) { return (floats + 63) / 64 * 64; }
// Whether K and V (and Q) as dense fp32 arrays, formed once by a launch of their own, beat rebuilding every tile from the factors in
// each workgroup: the rebuild grows with the rank and the blocks of rows that repeat it, the launch with the keys alone.  us, fused / dense,
// causal, 8 heads of 64 | 4 x 64 heads of 64 | 2 x 16 heads of 128:
//   rank 8: 40 rows over 300 keys 27.2 / 19.9 | 58.5 / 49.1 | 67.7 / 42.2; 200 x 200 19.6 / 19.0 | 60.3 / 46.8 | 49.9 / 30.5; 300 x 3000 183 / 76 | 1064 /
//     647 | 886 / 304; 700 x 700 50.0 / 28.6 | 329 / 175 | 272 / 124; but 17 x 300 27.2 / 19.5 | 31.2 / 36.4 | 66.9 / 36.4
//   rank 4: 40 x 300 19.5 / 18.8 | 39.0 / 47.9 | 45.9 / 39.4; 200 x 200 14.9 / 18.5 | 38.5 / 47.1 | 34.3 / 29.2; 40 x 2000 80 / 53 | 151 / 161 | 215 / 120; 300 x
//     300 19.4 / 19.0 | 87 / 76 | 47.3 / 40.9; 700 x 700 30.7 / 27.3 | 208 / 171 | 171 / 123
//   rank 3: 300 x 300 16.9 / 19.5 | 82 / 77 | 42.9 / 40.8; 100 x 1000 33.5 / 33.3 | 133 / 140 | 101 / 71; 700 x 700 27.3 / 26.7 | 190 / 170 | 156 / 123
//   rank 2: 700 x 700 23.7 / 26.9 | 176 / 173 | 139 / 124; 1500 x 1500 42.1 / 42.4 | 592 / 571 | 275 / 244, no mask 79 / 72 | 950 / 921 | 287 / 252; 4000 x 4000
//     202 / 176 | - | 796 / 742; 300 x 3000 70 / 75 | 586 / 615 | 411 / 298; 4 x 32 heads of 128 700 x 700 178 / 161, 4000 x 4000 3206 / 3138
//   rank 1: never (700 x 700 20.2 / 26.7 | 167 / 175 | 123 / 124)
bool f32_dense_pays(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D, int64_t rk) {
  const int64_t pairs = B * H;
  if (rk < 2 || lq <= 16) return false;
  if (rk == 2) return pairs <= 128 && lq >= (D == 128 ? 700 : 1500) && lk <= 5 * lq;  // beyond, 2 % for three arrays of O's size
  if (lq <= 32 && pairs > 64) return false;
  if (rk >= 8 || D == 128) return true;
  return pairs > 64 ? lq > 256 : lk * rk >= 2800;
}
}  // namespace
}  // namespace tpa

size_t tpa_prefill_f32_dense_bytes(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D, int64_t rk) {
  if (H % 8 != 0 || !tpa::f32_dense_pays(B, lq, lk, H, D, rk)) return 0;
  return (size_t)(tpa::dense_slot(B * lq * H * D) + 2 * tpa::dense_slot(B * lk * H * D)) * 4;
}

namespace tpa {
namespace {
F32Params params_of(const TpaFwdArgs* a) {  // on the factors as they are
  F32Params p{};
  p.qa = a->qa; p.qb = a->qb; p.ka = a->ka; p.kb = a->kb; p.va = a->va; p.vb = a->vb;
  p.qseg = a->q_segment_ids; p.kvseg = a->kv_segment_ids; p.kvlen = a->kv_lengths;
  p.o = static_cast<float*>(a->o); p.lse = a->lse;
  p.B = a->B; p.lq = a->lq; p.lk = a->lk; p.H = a->H; p.rq = a->rq; p.rk = a->rk;
  p.q_scale = a->sm_scale * kLog2e / (float)a->rq; p.causal = a->causal; p.coff = causal_offset_of(a);
  return p;
}
// and with Q (the scale in it), K and V as dense arrays of H * D floats a row
F32Params dense_params_of(const TpaFwdArgs* a, const float* qd, const float* kd, const float* vd) {
  F32Params p = params_of(a);
  const int64_t hd = (int64_t)a->H * a->dk;
  p.qa = p.ka = p.va = TpaFactor{nullptr, 0, 0, 0};
  p.qb = TpaFactor{qd, a->lq * hd, hd, 0};
  p.kb = TpaFactor{kd, a->lk * hd, hd, 0};
  p.vb = TpaFactor{vd, a->lk * hd, hd, 0};
  p.rq = p.rk = 1;
  p.q_scale = 1.f;
  return p;
}
}  // namespace
}  // namespace tpa

namespace tpa {
namespace {
// The same for one call, whose kernel, mask and ranks of Q are known: the us that dense arrays save there, from rank 3 on.  Against them
// stand the launch and the trip of K and V through memory, 0.2 us a MB; for them, every tile that a workgroup does not rebuild, as many as the longest
// walk of a block has or the rounds of average ones - in the kernel of 32 rows steps of its waves, 32 keys each, the first of which hides a part - and, in the
// others, Q, which they sum rank by rank.  Rank 3 costs less than its share.  Fitted to 2000 shapes of 17 to 2000 rows, ranks 3 to 16 (and 2, 4, 6, 16 of Q),
// within 1.2 us (32 rows) and 3 (256) for the half of them.  The line above alone took 100 of 1500 to the slower side by more than 2 %, with this 34, at the
// same gain over all (1.275).  fused / dense: 105 x 105, 3 x 16 heads of 128, rank 3 19.2 / 23.2; 100 x 100, 4 x 16, rank 3 19.6 / 24.8; 40 x 40, 12 x 32, rank 3 30.2 /
// 38.5; 307 x 307, 2 x 64 of 64, rank 4 47.5 / 56.4; 100 x 317 in documents of 161, 45 x 40 of 128, rank 3 381 / 463 (all stay fused); 33 x 1000, 2 x 16 heads of 64,
// rank 3 32.6 / 41.4 (does not); 25 x 25, 2 x 8, rank 4 of Q, 3 20.2 / 17.5; 200 x 200, 2 x 16 of 128, rank 4 34.3 / 29.2; 256 x 256, 8 x 32, rank 4 86.6 / 72.6; 256 x 1000, 4 x 32, rank 4 249 / 190.
double dense_saves_us(const TpaFwdArgs* a, int rows) {
  const int64_t D = a->dk, pairs = (int64_t)a->B * a->H, reach = keys_in_reach(a), nblk = ((int64_t)a->lq + rows - 1) / rows, wgs = nblk * pairs;
  if (nblk > 256) return 1e9;  // K and V of so many blocks are not made in vain
  const int64_t behind = a->causal ? causal_offset_of(a) + (a->causal == TPA_CAUSAL_BOTTOM_RIGHT ? a->lk - a->lq : 0) : a->lk;  // row i meets keys up to i + this
  const int64_t step = rows == 32 ? 32 * (D == 64 ? SplitLdsF32<64>::NW : SplitLdsF32<128>::NW) : 64;
  int64_t longest = 0, all = 0;
  for (int64_t i = 0; i < nblk; ++i) {
    const int64_t end = std::min(reach, std::max<int64_t>(0, (i + 1) * rows + behind)), steps = (end + step - 1) / step;
    longest = std::max(longest, steps);
    all += steps;
  }
  const double rounds = (double)((wgs + 255) / 256), rank = a->rk == 3 ? 2.7 : a->rk, mb = (double)(2 * pairs * reach * D) * 4e-6;
  double walk = std::max((double)longest, (double)all / nblk * rounds);
  // documents, whose lengths the host does not know, meet between as many keys as there are rows and all: half way
  if (a->kv_segment_ids && a->lk > a->lq && reach > 0) walk *= 0.5 + 0.5 * std::min(1., (double)(a->lq + 128) / (double)reach);
  if (rows == 32)
    return D == 64 ? (0.94 * walk - 0.30) * rank - 2.2 * wgs / 256 - 2.8 - 0.23 * mb : (1.63 * walk - 0.26) * rank - 3.3 * wgs / 256 - 2.2 - 0.24 * mb;
  if (rows == 128 && D == 128) return walk * (2.56 * rank - 2.8) + rounds * (2. * a->rq) - 25. - 0.05 * mb;
  return D == 64 ? walk * (0.69 * rank - 0.68) + rounds * (0.98 * a->rq - 3.6) - 8. - 0.16 * mb
                 : walk * (1.33 * rank - 1.2) + rounds * (1.63 * a->rq - 9.4) + 4.6 - 0.24 * mb;
}
}  // namespace
}  // namespace tpa

size_t tpa_prefill_f32_call_bytes(const TpaFwdArgs* a) {
  using namespace tpa;
  if (!tpa_recon_dense_qkv_f32_takes(a)) return 0;
  const size_t need = tpa_prefill_f32_dense_bytes(a->B, a->lq, a->lk, a->H, a->dk, a->rk);
  if (!need) return 0;
  const int rows = rows_per_workgroup(params_of(a), a->dk);
  if (a->rk > 2 && dense_saves_us(a, rows) < 0.5) return 0;
  // Rows of H * D floats reach the 2 GiB of the kernel of 32 rows before those of the factors do: a call that would fall from it to 256
  // rows stays on the factors (64 rows over 140 000 keys, 32 heads of 128, rank 4: 128 workgroups that share out the keys against 32 with
  // two of eight waves at work, and 4.6 GB).
  if (rows == 32 && !split_supported(dense_params_of(a, nullptr, nullptr, nullptr))) return 0;
  return need;
}

int tpa_prefill_f32_launch(const TpaFwdArgs* a, hipStream_t stream) {
  using namespace tpa;
  F32Params p = params_of(a);
  if (const size_t need = tpa_prefill_f32_call_bytes(a); need && a->workspace && !(reinterpret_cast<uintptr_t>(a->workspace) & 255) && a->workspace_bytes >= need) {
    const int64_t hd = (int64_t)a->H * a->dk;
    float* const kd = static_cast<float*>(a->workspace);
    float* const vd = kd + dense_slot(a->B * a->lk * hd);
    float* const qd = vd + dense_slot(a->B * a->lk * hd);
    if (const int rc = tpa_recon_dense_qkv_f32(a, qd, kd, vd, a->sm_scale * kLog2e, stream); rc != TPA_OK) return rc;
    p = dense_params_of(a, qd, kd, vd);
  }
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
  p.q_scale = a->sm_scale * kLog2e; p.causal = a->causal ? TPA_CAUSAL_TOP_LEFT : TPA_CAUSAL_NONE;
  return launch_any(p, a->dk, stream);
}
