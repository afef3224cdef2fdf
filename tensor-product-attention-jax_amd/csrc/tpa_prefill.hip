// Flash-style prefill for gfx950: bf16 MFMA contractions, fp32 online softmax.
//
// One workgroup = one (batch, head, block of 256 query rows): eight waves (two per SIMD, 256 registers
// each), a wave owns one block of 32 query rows.  At head size 64 it is 128 rows and four waves, two workgroups
// to a compute unit, where wants_four_waves() says so.
// Per tile of 64 keys the workgroup rebuilds the head's K and V
// tile from the rank factors (K = (1/R) sum_r a_r (x) b_r, tpa/tpa.py:364,417) straight out of
// coalesced 16-byte factor loads and stores it once, as bf16, in LDS.  Each wave then computes
//     S^T = K Q^T        (v_mfma_f32_32x32x16_bf16, A = K rows from LDS, B = Q kept in registers,
//                         Q pre-scaled by sm_scale*log2(e) and the accumulator started at minus
//                         the running reference, so the result is the exponent itself)
//     online softmax     (each lane holds 32 logits of ONE query row, so the row max, where one is
//                         taken, and sum are in-lane apart from one exchange with lane ^ 32)
//     O^T += V^T P^T     (A = V^T read with ds_read_b64_tr_b16 from row-major V, B = P^T, which
//                         is the S^T accumulator converted in place: no LDS round trip for P)
// with the deferred normalisation of flash attention (a reference m and a sum l per row), which
// is the normalise-every-step recurrence of tpa/tpa.py:389-424 in another order of operations.
// There is one workgroup barrier per tile (K tiles rotate through three LDS buffers, V tiles and the
// head factors through two).  Tiles that need no mask run a hand-scheduled loop generated by
// gen_prefill_loop.py (one for the dense loader, one for the rank-2 factor loader): the softmax of one
// piece of the key axis sits, instruction by instruction, behind the matrix instructions of the next
// piece's logits, and the loader's stores, the rebuild of the tiles ahead and the next loads behind the
// O^T instructions, so that no matrix instruction waits for vector work of its own iteration.  (A vector
// instruction issued while a matrix instruction of the same wave executes is nearly free on this
// hardware, whereas two waves of a SIMD that are both in a vector-only or both in a matrix-only phase
// just queue up; the dot instruction is the exception: it occupies the matrix pipe.)  Tile 0, masked tiles
// (diagonal, ragged, keys of other segments) and a wave's last tile run plain code (cold_compute).
// The dense flash baseline (tpa/mha.py:23-37) is the same kernel with a plain K/V loader.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "tpa_common.h"

namespace tpa {
namespace {

constexpr int kTK = 64;   // keys per tile
constexpr int kBQ = 256;  // query rows per workgroup: 8 blocks of 32, one per wave (or half of them, see wants_four_waves)

enum { LOAD_TPA_R2 = 0, LOAD_TPA_ANY = 1, LOAD_DENSE = 2 };

struct PrefillParams {
  TpaFactor qa, qb, ka, kb, va, vb;  // dense: qb/kb/vb hold q/k/v with stride_l = H*D, ptr at head 0
  const int32_t* qseg;   // [B, lq] or null
  const int32_t* kvseg;  // [B, lk] or null (both or neither)
  const int32_t* kvlen;  // [B] keys per batch entry, or null (= lk)
  uint16_t* o;
  float* lse;
  int B, lq, lk, H, rq, rk;
  float sm_scale;
  int causal;
  int coff;         // with causal: row i sees keys <= i + coff (0 = top-left aligned)
  int nqb;     // query blocks per (batch, head)
  int npairs;  // nqb * B
  int q_scaled;   // dense loader only: 1 = q already holds sm_scale * log2(e) * Q (it was reconstructed with that factor)
  int pair_groups; // dense loader only: groups of (batch, head) pairs of an XCD whose query blocks run side by side (see the kernel)
  int head_groups; // factor loaders only: see pair_of_workgroup
  // key ranges per query block (1: none).  nqb then counts (query block, range) and a workgroup's result goes, not
  // normalised, to part_o [S][B, lq, H, D] with the reference (log2 domain; -inf: no key seen) and the sum in part_ml
  int S;
  float* part_o;
  float2* part_ml;  // [S][B, lq, H]
  // dense loader with segment ids: 1 = the id window of a workgroup is an IdWindow in its first row of the output (written by the launch
  // that reconstructed Q, K, V, read before any of this workgroup's own results are written; no other workgroup writes that row of this head)
  int windows;
};

// LDS: three buffers of a K tile (tile j is read while tile j+1 is already there for waves that run
// a tile ahead with their logits, and tile j+2 is being written), two of a V tile, two slots of head
// factors and two of key segment ids: [K0][K1][K2][V0][V1][A0][A1][seg0][seg1], offsets in uint16 units.
template <int D>
struct Lds {
  static constexpr int KS = D + 8;   // K row stride (elements): 16-byte reads of 16 rows hit distinct banks
  static constexpr int VS = D + 32;  // V row stride: 4 consecutive rows of a transposed read hit distinct banks
  static constexpr int kK = kTK * KS;  // elements of one K buffer
  static constexpr int kV = kTK * VS;  // elements of one V buffer
  static constexpr int kA = 2 * kTK * 2;  // one slot of head factors: [K|V][token][rank 0|1]
  static constexpr int kSeg = 2 * kTK;    // one slot of key segment ids (int32), in uint16 units
  static constexpr int k_off(int buf) { return buf * kK; }
  static constexpr int v_off(int buf) { return 3 * kK + buf * kV; }
  static constexpr int a_off(int buf) { return 3 * kK + 2 * kV + buf * kA; }
  static constexpr int seg_off(int buf) { return 3 * kK + 2 * kV + 2 * kA + buf * kSeg; }
  static constexpr size_t kBytes = (3 * kK + 2 * (kV + kA + kSeg)) * sizeof(uint16_t);
};

// a0*b0 + a1*b1 on packed bf16 pairs, fp32 result.  Through the builtin on purpose: the dot
// instructions need software wait states before a dependent VALU instruction, which the compiler
// only inserts for instructions it selected itself (not for inline assembly).
__device__ __forceinline__ float dot2_bf16(uint32_t pair, uint32_t aa) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, aa), 0.f, false);
}

__device__ __forceinline__ float dot2_bf16_acc(uint32_t pair, uint32_t aa, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, aa), c, false);
}

// Workgroup barrier that waits for this wave's LDS traffic only.  __syncthreads() would also
// wait for the global loads of the next tile's factors, which are meant to stay in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// compile-time loop: f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N-1>{})
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}
template <int V>
using IC = std::integral_constant<int, V>;

// Batch entries by their lengths, longest first (equal ones in their order): lane = batch entry, B <= 64 (kMostOrdered are worth it).  A launch of several workgroups
// per compute unit ends with the last of them, so the long ones start first; every workgroup works the order out, as the lengths are known on the
// device only.
constexpr int kMostOrdered = 32;
struct LongestFirst {
  int len, B;
  __device__ __forceinline__ LongestFirst(const int32_t* kvlen, int B, int lk) : B(B) {
    const int lane = threadIdx.x & 63;
    len = max(0, min(kvlen[min(lane, B - 1)], lk));
  }
  // whether an order is worth anything: the lengths differ by more than an eighth of the longest
  __device__ __forceinline__ bool differ() const {
    const int longest = wave_max(len), shortest = wave_min(len);
    return scalar(longest - shortest > longest >> 3);
  }
  __device__ __forceinline__ int entry(int at) const {
    const int lane = threadIdx.x & 63;
    int ahead = 0;
    for (int e = 0; e < B; ++e) {
      const int other = __builtin_amdgcn_readlane(len, e);
      ahead += other > len || (other == len && e < lane);
    }
    return scalar(__builtin_ctzll(__ballot(lane < B && ahead == at)));
  }
};

// ORDER: batch entries of different lengths go longest first (an instance of its own: as a branch it cost every call 0.25 us, 1 x 500 tokens,
// 8 heads of 64 15.9 / 16.2)
template <int D, int LOADER, bool SEG, bool SPLIT, int NW, bool ORDER>
__global__ __launch_bounds__(NW * 64, 2) void prefill_kernel(PrefillParams pp) {
  // row blocks per wave: the per-wave state below is indexed by row block, and one is what fits 256 registers
  // (two per wave on four waves of 512 registers were slower: one wave per SIMD issues too slowly)
  constexpr int RB = 1;
  constexpr int NT = NW * 64, kRows = 32 * NW;  // query rows per workgroup
  using L = Lds<D>;
  constexpr int KS = L::KS, VS = L::VS;
  constexpr int CPR = D / 8;             // 16-byte chunks per row
  constexpr int TPP = NT / CPR;          // tokens per loader pass
  constexpr int NPASS = kTK / TPP;       // loader passes per tile and matrix
  static_assert(kTK % TPP == 0 && NPASS >= 1, "loader shape");
  constexpr int NKS = D / 16;            // k-steps of the QK^T contraction
  constexpr int NDB = D / 32;            // 32-row blocks of O^T
  constexpr float kSlack = 8.f;          // the reference only moves when a tile max exceeds it by 2^8

  // scalars out of the argument block (never take the address of the block itself)
  struct Fac { const uint16_t* ptr; int64_t stride_b; int stride_l, stride_r; };
  auto fac = [](const TpaFactor& f) { return Fac{static_cast<const uint16_t*>(f.ptr), f.stride_b, (int)f.stride_l, (int)f.stride_r}; };
  struct { Fac qa, qb, ka, kb, va, vb; const int32_t* qseg; const int32_t* kvseg; const int32_t* kvlen; uint16_t* o; float* lse; int B, lq, lk, H, rq, rk; float sm_scale; int causal, coff, nqb, npairs, q_scaled, pair_groups, head_groups, S; } const p = {
      fac(pp.qa), fac(pp.qb), fac(pp.ka), fac(pp.kb), fac(pp.va), fac(pp.vb), pp.qseg, pp.kvseg, pp.kvlen, pp.o, pp.lse, pp.B, pp.lq, pp.lk, pp.H, pp.rq, pp.rk,
      pp.sm_scale, pp.causal, pp.causal ? pp.coff : 0, pp.nqb, pp.npairs, pp.q_scaled, pp.pair_groups, pp.head_groups, SPLIT ? pp.S : 1};

  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  auto lds_k = [&](int buf) __attribute__((always_inline)) { return smem + L::k_off(buf); };    // [kTK][KS]
  auto lds_v = [&](int buf) __attribute__((always_inline)) { return smem + L::v_off(buf); };    // [kTK][VS]
  auto lds_a = [&](int buf) __attribute__((always_inline)) { return smem + L::a_off(buf); };    // [K|V][kTK][2]
  auto lds_seg = [&](int buf) __attribute__((always_inline)) { return reinterpret_cast<int32_t*>(smem + L::seg_off(buf)); };  // [kTK]

  // ---- which (query block, batch, head); (block, batch) pairs are ordered heaviest (last causal block) first
  const int id = blockIdx.x;
  int h, b, qblk;
  if constexpr (LOADER == LOAD_DENSE) {
    // Dense K and V belong to one (batch, head): what workgroups can share is the K/V stream of
    // their head.  An XCD therefore owns whole (batch, head) pairs and runs them in groups of
    // pairs: the query blocks of a group heaviest first, the same block of the group's
    // pairs side by side.  The 32 workgroups that are resident together on an XCD are then
    // neighbouring query blocks of a few pairs, which walk the same tiles at about the same time and
    // find them in that XCD's L2 (with every pair of the XCD in one group and many pairs, the resident
    // workgroups would all belong to different pairs and every tile would come from memory).
    int bh, rank;
    if (!pair_in_group(id, p.B * p.H, p.pair_groups, p.nqb, bh, rank)) return;
    qblk = p.nqb - 1 - rank;
    b = bh / p.H;
    h = bh % p.H;
    if constexpr (ORDER) b = LongestFirst(p.kvlen, p.B, p.lk).entry(b);
  } else {
    // Where the lengths differ, all heads of an entry on one XCD, or of the same entries in every round, would leave the XCDs of the short
    // ones idle: the heads then go in eight groups, one per XCD, and an entry's blocks side by side.
    int pair;
    bool differ = false;
    if constexpr (ORDER) {
      const LongestFirst order(p.kvlen, p.B, p.lk);
      differ = order.differ();
      if (differ) {
        if (!pair_of_workgroup(id, p.npairs, p.H, p.B, 8, pair, h)) return;
        qblk = p.nqb - 1 - pair % p.nqb;
        b = order.entry(pair / p.nqb);
      }
    }
    if (!differ) {
      if (!pair_of_workgroup(id, p.npairs, p.H, p.B, p.head_groups, pair, h)) return;
      qblk = p.nqb - 1 - pair / p.B;
      b = pair % p.B;
    }
  }

  int range = 0;
  if constexpr (SPLIT) {
    range = qblk % p.S;
    qblk /= p.S;
  }

  const int tid = threadIdx.x;
  const int w = scalar(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
  const int q0 = qblk * kRows;
  // row block r of this wave within the workgroup's (one per wave)
  int rblk[RB], wrow0[RB], qrow[RB], qrow_ld[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    rblk[r] = w;
    wrow0[r] = q0 + 32 * rblk[r];  // first query row of the block
    qrow[r] = wrow0[r] + i;        // this lane's row in it
    qrow_ld[r] = min(qrow[r], p.lq - 1);
  }
  const float c = (LOADER == LOAD_DENSE && p.q_scaled) ? 1.f : p.sm_scale * kLog2e;

  // ---- Q fragments (B operand of S^T = K Q^T), scaled by c: lane (i, g) holds
  // c * Q[qrow[r]][16ks + 8g + 0..7]
  bf16x8 qf[RB][NKS];
  auto build_q = [&]() __attribute__((always_inline)) {
    // the dense loader serves dense attention and factored attention whose Q, K and V were
    // reconstructed beforehand (Q with its scale factor, so that it is rounded to bf16 once)
    if constexpr (LOADER == LOAD_DENSE) {
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const uint16_t* qp = p.qb.ptr + b * p.qb.stride_b + (int64_t)qrow_ld[r] * p.qb.stride_l + (int64_t)h * D;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          const u32x4 raw = *reinterpret_cast<const u32x4*>(qp + 16 * ks + 8 * g);
          u32x4 sc;
#pragma unroll
          for (int j = 0; j < 4; ++j) sc[j] = pack_bf16(bf16lo_to_f32(raw[j]) * c, bf16hi_to_f32(raw[j]) * c);
          qf[r][ks] = __builtin_bit_cast(bf16x8, sc);
        }
      }
    } else {
      // One rank at a time through LDS: the workgroup copies the kRows x D slab qb[q0.., r, :] with
      // coalesced 16-byte loads (each row is read once, not once per lane pair), then every lane
      // picks up its own row's fragments.  The next rank's loads are in flight meanwhile.
      constexpr int QS = D + 8;                  // row stride in LDS (elements)
      constexpr int CH = kRows * CPR / NT;         // 16-byte chunks per thread and rank
      uint16_t* const qs = smem;                 // [kRows][QS]
      uint16_t* const qas = smem + kRows * QS;     // [kRows] head factors of this rank
      static_assert((kRows * QS + kRows) * sizeof(uint16_t) <= L::kBytes, "Q staging fits the K/V buffers");
      const uint16_t* qb_b = p.qb.ptr + b * p.qb.stride_b;
      const uint16_t* qa_b = p.qa.ptr + b * p.qa.stride_b + h;
      u32x4 nxt[CH];
      uint32_t a_nxt = 0;
      auto load_rank = [&](int r) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < CH; ++q) {
          const int chunk = q * NT + tid, row = chunk / CPR, cc = chunk % CPR;
          const int grow = min(q0 + row, p.lq - 1);
          nxt[q] = *reinterpret_cast<const u32x4*>(qb_b + (int64_t)grow * p.qb.stride_l + r * p.qb.stride_r + 8 * cc);
        }
        if (tid < kRows) a_nxt = qa_b[(int64_t)min(q0 + tid, p.lq - 1) * p.qa.stride_l + r * p.qa.stride_r];
      };
      float acc[RB][NKS][8];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[rb][ks][j] = 0.f;
      load_rank(0);
      for (int r = 0; r < p.rq; ++r) {
#pragma unroll
        for (int q = 0; q < CH; ++q) {
          const int chunk = q * NT + tid, row = chunk / CPR, cc = chunk % CPR;
          *reinterpret_cast<u32x4*>(qs + row * QS + 8 * cc) = nxt[q];
        }
        if (tid < kRows) qas[tid] = (uint16_t)a_nxt;
        if (r + 1 < p.rq) load_rank(r + 1);
        lds_barrier();
        // a * b[d] for a packed pair (b[d], b[d+1]) is one dot instruction with (a, 0) or (0, a):
        // no unpacking, and the dot unit is idle here anyway
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          const int row = 32 * rblk[rb] + i;
          const uint32_t a_lo = qas[row], a_hi = a_lo << 16;
#pragma unroll
          for (int ks = 0; ks < NKS; ++ks) {
            const u32x4 bv = *reinterpret_cast<const u32x4*>(qs + row * QS + 16 * ks + 8 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              uint32_t pair = bv[j];
              asm volatile("" : "+v"(pair));  // keeps the compiler from taking element 0 of the vector for every j
              acc[rb][ks][2 * j] = dot2_bf16_acc(pair, a_lo, acc[rb][ks][2 * j]);
              acc[rb][ks][2 * j + 1] = dot2_bf16_acc(pair, a_hi, acc[rb][ks][2 * j + 1]);
            }
          }
        }
        lds_barrier();  // everyone has read this rank before the next one overwrites it
      }
      const float scale = c / (float)p.rq;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          u32x4 packed;
#pragma unroll
          for (int j = 0; j < 4; ++j) packed[j] = pack_bf16(acc[rb][ks][2 * j] * scale, acc[rb][ks][2 * j + 1] * scale);
          qf[rb][ks] = __builtin_bit_cast(bf16x8, packed);
        }
    }
  };

  // ---- key range [kpos0, kend) this workgroup visits; tiles are counted from kpos0
  int kpos0 = 0;
  const int len_b = p.kvlen ? max(0, min(p.kvlen[b], p.lk)) : p.lk;  // keys of this batch entry
  // causal offset of this batch entry: counted from the end of its keys where the caller aligns the last
  // query with the last key
  const int coff = p.coff + (p.causal == TPA_CAUSAL_BOTTOM_RIGHT ? len_b - p.lq : 0);
  int kend = p.causal ? min(len_b, min(q0 + kRows, p.lq) + coff) : len_b;
  if constexpr (SPLIT) {  // this workgroup's share of the block's tiles
    const int all = kend > 0 ? (kend + kTK - 1) / kTK : 0;
    const int t0 = (int)((int64_t)all * range / p.S), t1 = (int)((int64_t)all * (range + 1) / p.S);
    if (t0 == t1) {
      if (tid < kRows && q0 + tid < p.lq) pp.part_ml[(((int64_t)range * p.B + b) * p.lq + q0 + tid) * p.H + h] = float2{-INFINITY, 0.f};
      return;
    }
    kpos0 = t0 * kTK;
    kend = min(kend, t1 * kTK);
  } else if (kend <= 0) {  // no key at all: the rows end as NaN / -inf (tpa/tpa.py:437-439)
#pragma unroll
    for (int r = 0; r < RB; ++r)
      if (qrow[r] < p.lq) {
        uint16_t* op = p.o + (((int64_t)b * p.lq + qrow[r]) * p.H + h) * D;
        const u32x4 nan4 = {0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u};
#pragma unroll
        for (int cch = 0; cch < D / 16; ++cch) *reinterpret_cast<u32x4*>(op + 16 * cch + 8 * g) = nan4;
        if (p.lse && g == 0) p.lse[((int64_t)b * p.H + h) * p.lq + qrow[r]] = -INFINITY;
      }
    return;
  }
  bool seg_pure = false;  // every visited key from the second tile on carries the rows' one segment id
  if constexpr (SEG) {
    // Packed sequences: a key can only be visible to this block if its id lies within the
    // [min, max] of the block's query ids.  The workgroup scans the key ids once, keeps the first
    // and the last such key, and visits only the tiles between them (exact for ids that do not
    // decrease along the sequence; any other id pattern just visits more tiles, the mask itself
    // is applied per key as before).  If the rows share one id and the keys with that id form one
    // contiguous run, the tiles inside the run need no segment mask at all.
    int lo, hi, cnt;
    int32_t qmin, qmax;
    if (LOADER == LOAD_DENSE && pp.windows) {
      const IdWindow* const win = reinterpret_cast<const IdWindow*>(p.o + (((int64_t)b * p.lq + q0) * p.H + h) * D);
      lo = scalar(win->first); hi = scalar(win->last); cnt = scalar(win->count); qmin = scalar(win->least); qmax = scalar(win->most);
    } else id_window<NT>(p.qseg + (int64_t)b * p.lq + q0, min(kRows, p.lq - q0), p.kvseg + (int64_t)b * p.lk, kend, reinterpret_cast<int32_t*>(smem), tid, lo, hi, cnt, qmin, qmax);
    if (hi >= 0) {
      kpos0 = lo / kTK * kTK;
      kend = hi + 1;
      seg_pure = scalar(qmin == qmax && cnt == hi - lo + 1);
    } else {
      kend = min(kend, kTK);  // nothing visible: one (fully masked) tile, the rows end as NaN / -inf
    }
  }
  kpos0 = scalar(kpos0);
  kend = scalar(kend);
  const int lk_r = kend - kpos0;          // keys counted from kpos0
  const int ntiles = (lk_r + kTK - 1) / kTK;
  const int last = ntiles - 1;
  // first row of each of this wave's row blocks and this lane's row in it on that scale, shifted by
  // the causal offset: row x sees keys up to x_r, which is negative for a row that sees none;
  // last tile the block needs under the causal mask (its rows: wrow0 .. wrow0 + 31)
  int wrow_r[RB], qrow_r[RB], wave_last_tile[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    wrow_r[r] = wrow0[r] + coff - kpos0;
    qrow_r[r] = qrow[r] + coff - kpos0;
    wave_last_tile[r] = p.causal ? min(last, max(wrow_r[r] + 31, 0) / kTK) : last;
  }

  // ---- loader: this thread rebuilds chunk lc (8 elements) of token lt (+ TPP per pass).
  // Addresses are a uniform (scalar) tile base plus a per-thread 32-bit element offset.
  const int lt = tid / CPR, lc = tid % CPR;
  u32x4 kreg[NPASS][2], vreg[NPASS][2];  // LOAD_TPA_R2: two ranks; LOAD_DENSE: [0] only

  // all key-side bases point at key kpos0
  const uint16_t* const kb_b = p.kb.ptr + b * p.kb.stride_b + (int64_t)kpos0 * p.kb.stride_l + (LOADER == LOAD_DENSE ? (int64_t)h * D : 0);
  const uint16_t* const vb_b = p.vb.ptr + b * p.vb.stride_b + (int64_t)kpos0 * p.vb.stride_l + (LOADER == LOAD_DENSE ? (int64_t)h * D : 0);
  const uint16_t* const ka_b = p.ka.ptr + b * p.ka.stride_b + (int64_t)kpos0 * p.ka.stride_l + h;
  const uint16_t* const va_b = p.va.ptr + b * p.va.stride_b + (int64_t)kpos0 * p.va.stride_l + h;

  // B-factor loads of one matrix (K or V) for one tile into registers.  They are raw buffer
  // loads: resource = this batch entry's matrix (in scalar registers), scalar offset = (tile,
  // pass, rank), vector offset = this thread's fixed place inside a pass - no vector instruction
  // is spent on addresses, and rows past the end of the sequence read as zero (the range check
  // of the resource), so a ragged last tile needs no clamping.
  constexpr int kRsrcFlags = 0x00020000;  // raw 32-bit data format
  const int k_rows_bytes = ((lk_r - 1) * p.kb.stride_l + (LOADER == LOAD_TPA_R2 ? p.kb.stride_r : 0) + D) * 2;
  const int v_rows_bytes = ((lk_r - 1) * p.vb.stride_l + (LOADER == LOAD_TPA_R2 ? p.vb.stride_r : 0) + D) * 2;
  const __amdgpu_buffer_rsrc_t kb_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kb_b), 0, k_rows_bytes, kRsrcFlags);
  const __amdgpu_buffer_rsrc_t vb_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(vb_b), 0, v_rows_bytes, kRsrcFlags);
  const int kvoff = (lt * p.kb.stride_l + 8 * lc) * 2, vvoff = (lt * p.vb.stride_l + 8 * lc) * 2;
  auto issue_into = [&](u32x4 (&regs)[NPASS][2], auto is_v_c, int tile) __attribute__((always_inline)) {
    constexpr bool is_v = decltype(is_v_c)::value;
    if constexpr (LOADER == LOAD_TPA_ANY) return;
    const int sl = is_v ? p.vb.stride_l : p.kb.stride_l, sr = is_v ? p.vb.stride_r : p.kb.stride_r;
#pragma unroll
    for (int ps = 0; ps < NPASS; ++ps) {
      const int soff = (tile * kTK + ps * TPP) * sl * 2;  // uniform
      regs[ps][0] = __builtin_amdgcn_raw_buffer_load_b128(is_v ? vb_rs : kb_rs, is_v ? vvoff : kvoff, soff, 0);
      if constexpr (LOADER == LOAD_TPA_R2) regs[ps][1] = __builtin_amdgcn_raw_buffer_load_b128(is_v ? vb_rs : kb_rs, is_v ? vvoff : kvoff, soff + 2 * sr, 0);
    }
  };
  auto issue = [&](auto is_v_c, int tile) __attribute__((always_inline)) {
    if constexpr (decltype(is_v_c)::value) issue_into(vreg, is_v_c, tile); else issue_into(kreg, is_v_c, tile);
  };
  using IsK = std::integral_constant<bool, false>;
  using IsV = std::integral_constant<bool, true>;

  // Head factors (LOAD_TPA_R2): a thread fetches one value a[matrix][token][rank], matrix = (tid % 256) / 128
  // (0: K of tile kt, 1: V of tile vt), token = (tid / 2) % 64, rank = tid % 2, and parks it in a register
  // until it is stored into an LDS slot one iteration later.  Where there are eight, waves 4-7 repeat what waves 0-3 do (same
  // values to the same addresses), so that all run one instruction stream.
  uint32_t a_pending = 0;
  const int a_idx = tid & (4 * kTK - 1);
  const int a_mat = scalar(a_idx / (2 * kTK)), a_tok = (a_idx >> 1) % kTK, a_rank = a_idx & 1;
  const int ka_bytes = ((lk_r - 1) * p.ka.stride_l + p.ka.stride_r + 1) * 2, va_bytes = ((lk_r - 1) * p.va.stride_l + p.va.stride_r + 1) * 2;
  const __amdgpu_buffer_rsrc_t ka_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(ka_b), 0, ka_bytes, kRsrcFlags);
  const __amdgpu_buffer_rsrc_t va_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(va_b), 0, va_bytes, kRsrcFlags);
  const int ka_voff = (a_tok * p.ka.stride_l + a_rank * p.ka.stride_r) * 2, va_voff = (a_tok * p.va.stride_l + a_rank * p.va.stride_r) * 2;
  auto issue_a = [&](int kt, int vt) __attribute__((always_inline)) {
    if constexpr (LOADER != LOAD_TPA_R2) return;
    // waves 0, 1 (4, 5) fetch K's head factors, waves 2, 3 (6, 7) V's (uniform per wave); tokens past the end read as 0
    if (a_mat == 0) a_pending = __builtin_amdgcn_raw_buffer_load_b16(ka_rs, ka_voff, kt * kTK * p.ka.stride_l * 2, 0);
    else a_pending = __builtin_amdgcn_raw_buffer_load_b16(va_rs, va_voff, vt * kTK * p.va.stride_l * 2, 0);
  };
  auto store_a = [&](int slot_idx) __attribute__((always_inline)) {
    if constexpr (LOADER != LOAD_TPA_R2) return;
    // stored halved (exact in bf16): the 1/R of the reconstruction with R = 2
    lds_a(slot_idx)[a_idx] = (uint16_t)(pack_bf16(bf16lo_to_f32(a_pending) * 0.5f, 0.f));
  };

  // Key segment ids (packed sequences, tpa/tpa.py:369-375): the threads of one wave (wave 4 where
  // there are eight, else wave 0) fetch one id of a tile each, park it in a register and store it
  // into an LDS slot one iteration later, like the head factors; slot j&1 holds the ids of tile j
  // during iteration j.
  constexpr bool has_seg = SEG;  // a kernel of its own: the mask code slows the others down even when skipped
  constexpr int kSegWave = NW > 4 ? 4 : 0;
  int32_t seg_pending = 0;
  auto issue_seg = [&](int tile) __attribute__((always_inline)) {
    if constexpr (has_seg)
      if (w == kSegWave) seg_pending = p.kvseg[(int64_t)b * p.lk + kpos0 + min(tile * kTK + l, lk_r - 1)];
  };
  auto store_seg = [&](int slot_idx) __attribute__((always_inline)) {
    if constexpr (has_seg)
      if (w == kSegWave) lds_seg(slot_idx)[l] = seg_pending;
  };
  int32_t qseg[RB] = {};
  if constexpr (has_seg) {
#pragma unroll
    for (int r = 0; r < RB; ++r) qseg[r] = p.qseg[(int64_t)b * p.lq + qrow_ld[r]];
  }
  const TileIds<has_seg, RB> ids_of_wave(qseg);
  bool masked_ids = false;  // tile j needs its segment mask for this wave's rows

  // (a0/2)*b0[d] + (a1/2)*b1[d] for 8 consecutive d; aa = packed (a0/2, a1/2): fetch_aa hands out
  // halved head factors.
  // Three short assembly pieces, so that they can sit between MFMAs: 8 v_perm_b32 (pair b0[d]
  // with b1[d]), 8 v_dot2_f32_bf16 (the VOP3P form with a zero addend, so no accumulator has to
  // be cleared first) and 4 v_cvt_pk_bf16_f32.  A dot result may only be read by another
  // vector-ALU instruction three wait states later and the hardware does not interlock; the
  // s_nop at the head of the last piece guarantees them whatever was scheduled in between.
  struct Chunk { uint32_t t0, t1, t2, t3, t4, t5, t6, t7; };
  auto rebuild_perm = [&](Chunk& c_, const u32x4& b0, const u32x4& b1) __attribute__((always_inline)) {
    const uint32_t sel_lo = 0x05040100u, sel_hi = 0x07060302u;
    asm volatile(
        "v_perm_b32 %0, %9, %8, %16\n\t"   // (b0[0], b1[0])
        "v_perm_b32 %1, %9, %8, %17\n\t"   // (b0[1], b1[1])
        "v_perm_b32 %2, %11, %10, %16\n\t"
        "v_perm_b32 %3, %11, %10, %17\n\t"
        "v_perm_b32 %4, %13, %12, %16\n\t"
        "v_perm_b32 %5, %13, %12, %17\n\t"
        "v_perm_b32 %6, %15, %14, %16\n\t"
        "v_perm_b32 %7, %15, %14, %17"
        : "=&v"(c_.t0), "=&v"(c_.t1), "=&v"(c_.t2), "=&v"(c_.t3), "=&v"(c_.t4), "=&v"(c_.t5), "=&v"(c_.t6), "=&v"(c_.t7)
        : "v"(b0[0]), "v"(b1[0]), "v"(b0[1]), "v"(b1[1]), "v"(b0[2]), "v"(b1[2]), "v"(b0[3]), "v"(b1[3]), "s"(sel_lo), "s"(sel_hi));
  };
  auto rebuild_dot = [&](Chunk& c_, uint32_t aa) __attribute__((always_inline)) {
    asm volatile(
        "v_dot2_f32_bf16 %0, %0, %8, 0\n\t"
        "v_dot2_f32_bf16 %1, %1, %8, 0\n\t"
        "v_dot2_f32_bf16 %2, %2, %8, 0\n\t"
        "v_dot2_f32_bf16 %3, %3, %8, 0\n\t"
        "v_dot2_f32_bf16 %4, %4, %8, 0\n\t"
        "v_dot2_f32_bf16 %5, %5, %8, 0\n\t"
        "v_dot2_f32_bf16 %6, %6, %8, 0\n\t"
        "v_dot2_f32_bf16 %7, %7, %8, 0"
        : "+v"(c_.t0), "+v"(c_.t1), "+v"(c_.t2), "+v"(c_.t3), "+v"(c_.t4), "+v"(c_.t5), "+v"(c_.t6), "+v"(c_.t7)
        : "v"(aa));
  };
  auto rebuild_cvt = [&](Chunk& c_) __attribute__((always_inline)) -> u32x4 {
    asm volatile(
        "s_nop 2\n\t"
        "v_cvt_pk_bf16_f32 %0, %0, %1\n\t"
        "v_cvt_pk_bf16_f32 %2, %2, %3\n\t"
        "v_cvt_pk_bf16_f32 %4, %4, %5\n\t"
        "v_cvt_pk_bf16_f32 %6, %6, %7"
        : "+v"(c_.t0), "+v"(c_.t1), "+v"(c_.t2), "+v"(c_.t3), "+v"(c_.t4), "+v"(c_.t5), "+v"(c_.t6), "+v"(c_.t7));
    return u32x4{c_.t0, c_.t2, c_.t4, c_.t6};
  };
  // halve a packed (a0, a1) pair (exact in bf16): 1/R with R = 2
  auto halve_pair = [&](uint32_t aa_bits) __attribute__((always_inline)) -> uint32_t {
    return pack_bf16(bf16lo_to_f32(aa_bits) * 0.5f, bf16hi_to_f32(aa_bits) * 0.5f);
  };
  auto rebuild_r2 = [&](const u32x4& b0, const u32x4& b1, uint32_t aa_bits) __attribute__((always_inline)) -> u32x4 {
    Chunk c_;
    rebuild_perm(c_, b0, b1);
    rebuild_dot(c_, aa_bits);
    return rebuild_cvt(c_);
  };

  auto rebuild_any = [&](const uint16_t* bptr, const uint16_t* aptr, int b_stride_r, int a_stride_r) __attribute__((always_inline)) -> u32x4 {
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
    for (int r = 0; r < p.rk; ++r) {
      const float a = bf16bits_to_f32(aptr[r * a_stride_r]);
      const u32x4 bv = *reinterpret_cast<const u32x4*>(bptr + r * b_stride_r);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[2 * j] += a * bf16lo_to_f32(bv[j]);
        acc[2 * j + 1] += a * bf16hi_to_f32(bv[j]);
      }
    }
    const float inv = 1.f / (float)p.rk;
    u32x4 out;
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = pack_bf16(acc[2 * j] * inv, acc[2 * j + 1] * inv);
    return out;
  };

  // Head factors of this thread's tokens for one matrix of tile `tile`, as packed (a0, a1) pairs:
  // from the LDS slot ([K|V][token][rank]) or, with a_slot == nullptr, from global memory.
  auto fetch_aa = [&](auto is_v_c, int tile, const uint16_t* a_slot, uint32_t (&aa)[NPASS]) __attribute__((always_inline)) {
    constexpr bool is_v = decltype(is_v_c)::value;
    if constexpr (LOADER != LOAD_TPA_R2) return;
    const uint16_t* ab = is_v ? va_b : ka_b;
    const int a_sl = is_v ? p.va.stride_l : p.ka.stride_l, a_sr = is_v ? p.va.stride_r : p.ka.stride_r;
#pragma unroll
    for (int ps = 0; ps < NPASS; ++ps) {
      const int t = ps * TPP + lt;
      if (a_slot) {
        aa[ps] = *reinterpret_cast<const uint32_t*>(a_slot + (is_v ? 2 * kTK : 0) + 2 * t);
      } else {
        const int tok = min(tile * kTK + t, lk_r - 1);
        const uint32_t a0 = ab[(int64_t)tok * a_sl], a1 = ab[(int64_t)tok * a_sl + a_sr];
        aa[ps] = halve_pair(a0 | (a1 << 16));
      }
    }
  };

  // Rebuild one matrix of tile `tile` from the registers `issue` filled and store it in LDS.
  auto commit_from = [&](const u32x4 (&regs)[NPASS][2], auto is_v_c, int tile, const uint32_t (&aa)[NPASS]) __attribute__((always_inline)) {
    constexpr bool is_v = decltype(is_v_c)::value;
    const uint16_t* bb = is_v ? vb_b : kb_b;
    const uint16_t* ab = is_v ? va_b : ka_b;
    const int b_sl = is_v ? p.vb.stride_l : p.kb.stride_l, b_sr = is_v ? p.vb.stride_r : p.kb.stride_r;
    const int a_sl = is_v ? p.va.stride_l : p.ka.stride_l, a_sr = is_v ? p.va.stride_r : p.ka.stride_r;
    uint16_t* dst = is_v ? lds_v(tile & 1) : lds_k(tile % 3);
    constexpr int row_stride = is_v ? VS : KS;
#pragma unroll
    for (int ps = 0; ps < NPASS; ++ps) {
      const int t = ps * TPP + lt;
      u32x4 val;
      if constexpr (LOADER == LOAD_TPA_R2) {
        val = rebuild_r2(regs[ps][0], regs[ps][1], aa[ps]);
      } else if constexpr (LOADER == LOAD_TPA_ANY) {
        const int tok = min(tile * kTK + t, lk_r - 1);
        val = rebuild_any(bb + (int64_t)tok * b_sl + 8 * lc, ab + (int64_t)tok * a_sl, b_sr, a_sr);
      } else {
        val = regs[ps][0];
      }
      *reinterpret_cast<u32x4*>(dst + t * row_stride + 8 * lc) = val;
    }
  };
  auto commit = [&](auto is_v_c, int tile, const uint32_t (&aa)[NPASS]) __attribute__((always_inline)) {
    if constexpr (decltype(is_v_c)::value) commit_from(vreg, is_v_c, tile, aa); else commit_from(kreg, is_v_c, tile, aa);
  };

  // ---- per-wave state, one set per row block r (always indexed with compile-time constants)
  f32x16 o[RB][NDB];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[r][db][v] = 0.f;
  f32x16 s[RB][2];      // exponents x*c - mref of the tile in flight: two 32-key blocks per row block
  // P^T of the tile (packed bf16 pairs, the B operands of the four 16-key steps of O^T) is kept
  // in the registers of the logits it was made from: fragment k = s[r][k / 2][4 (k % 2) .. + 3]
  auto pf_set = [&](auto r_c, auto mb_c, auto idx_c, uint32_t bits) __attribute__((always_inline)) {
    s[decltype(r_c)::value][decltype(mb_c)::value][decltype(idx_c)::value] = __uint_as_float(bits);
  };
  auto pf_get = [&](auto r_c, auto kk_c) __attribute__((always_inline)) -> bf16x8 {
    constexpr int r = decltype(r_c)::value, kk = decltype(kk_c)::value, mb = kk / 2, h4 = 4 * (kk % 2);
    const u32x4 w4 = {__float_as_uint(s[r][mb][h4]), __float_as_uint(s[r][mb][h4 + 1]), __float_as_uint(s[r][mb][h4 + 2]), __float_as_uint(s[r][mb][h4 + 3])};
    return __builtin_bit_cast(bf16x8, w4);
  };
  float mref[RB];       // reference (log2 domain, includes c) of row qrow[r]
  // -mref in all 16 registers of an accumulator tuple: the addend of the first S^T MFMA of a
  // block, so the contraction lands on x*c - mref.  Rewritten only when the reference moves.
  f32x16 nmref[RB];
  float lsum[RB];       // this lane's share of sum exp2(x*c - mref)
  bool seen[RB];        // the row has met a visible key (its reference is set)
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    mref[r] = 0.f;
    lsum[r] = 0.f;
    seen[r] = false;
#pragma unroll
    for (int v = 0; v < 16; ++v) nmref[r][v] = 0.f;
  }
  auto refresh_nmref = [&](auto r_c) __attribute__((always_inline)) {
    constexpr int r = decltype(r_c)::value;
#pragma unroll
    for (int v = 0; v < 16; ++v) nmref[r][v] = -mref[r];
  };
  const int lp = l & 15, dhalf = (l >> 4) & 1;

  // masks + online softmax of tile `tile` for row block r (32 of the 64 logits of row qrow[r] live in this lane)
  auto do_softmax = [&](int tile, auto r_c) __attribute__((always_inline)) {
    constexpr int r = decltype(r_c)::value;
    const int k0 = tile * kTK;
    // keys beyond lk, and keys after the query under the causal mask
    const bool need_mask = (k0 + kTK > lk_r) || (p.causal && (k0 + kTK - 1 > wrow_r[r]));
    if (need_mask) {
      const int limit = p.causal ? min(qrow_r[r], lk_r - 1) : lk_r - 1;  // largest visible key index
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int t = k0 + 32 * mb + 8 * (v >> 2) + 4 * g + (v & 3);
          if (t > limit) s[r][mb][v] = -INFINITY;
        }
    }
    // keys of another segment (tpa/tpa.py:369-375)
    if (has_seg && masked_ids) {
      const int32_t* slot = lds_seg(tile & 1);
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          const int4 ids = *reinterpret_cast<const int4*>(slot + 32 * mb + 8 * vq + 4 * g);
          if (ids.x != qseg[r]) s[r][mb][4 * vq] = -INFINITY;
          if (ids.y != qseg[r]) s[r][mb][4 * vq + 1] = -INFINITY;
          if (ids.z != qseg[r]) s[r][mb][4 * vq + 2] = -INFINITY;
          if (ids.w != qseg[r]) s[r][mb][4 * vq + 3] = -INFINITY;
        }
    }
    float tmax = s[r][0][0];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int v = 0; v < 16; ++v) tmax = fmaxf(tmax, s[r][mb][v]);
    tmax = halves_max(tmax);
    const bool first = !seen[r] && tmax > -INFINITY;  // first tile with a visible key for this row
    const bool up = seen[r] && tmax > kSlack;         // rare: the row's max left the slack
    if (__any(first || up)) {
      // a first tile sets the reference (nothing accumulated yet, so nothing to rescale); later
      // the references move up and O and the row sums are rescaled.  The reference is always a whole
      // number: every exponent 2^(x - mref) then has the mantissa of 2^x itself, so which tile set or
      // moved the reference changes no rounding of P (and all rescaling is by exact powers of two)
      const float delta = (first || up) ? __builtin_ceilf(tmax) : 0.f;
      const float alpha = first ? 1.f : __builtin_amdgcn_exp2f(-delta);
      mref[r] += delta;
      refresh_nmref(r_c);
      lsum[r] *= alpha;
      if (__any(up)) {
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
#pragma unroll
          for (int v = 0; v < 16; ++v) o[r][db][v] *= alpha;
        }
      }
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) s[r][mb][v] -= delta;
      seen[r] = seen[r] || first;
    }
    static_for<4>([&](auto k_c) __attribute__((always_inline)) {
      constexpr int k = decltype(k_c)::value, mb = k / 2, half = k % 2;
      u32x4 pk;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p0 = __builtin_amdgcn_exp2f(s[r][mb][8 * half + 2 * j]);
        const float p1 = __builtin_amdgcn_exp2f(s[r][mb][8 * half + 2 * j + 1]);
        lsum[r] += p0 + p1;
        pk[j] = pack_bf16(p0, p1);
      }
      static_for<4>([&](auto j_c) __attribute__((always_inline)) {
        pf_set(r_c, IC<mb>{}, IC<4 * half + decltype(j_c)::value>{}, pk[decltype(j_c)::value]);
      });
    });
  };

  // ---------------------------------------------------------------------------------------
  // Main loop.  K runs one tile ahead of V, so that a wave may compute the logits of tile j+1
  // while it is still busy with the softmax of tile j.  Invariant at entry of iteration j: K tiles
  // j and j+1 are in LDS buffers j%3 and (j+1)%3, V tile j in buffer j&1; kreg holds the B factors
  // of K tile j+2 and vreg those of V tile j+1; head-factor slot j&1 holds those of K tile j+2 and
  // V tile j+1, a_pending (waves 0-3) those of K tile j+3 / V tile j+2 (tile indices clamped to
  // the last tile).  An iteration computes S^T = K Q^T, the softmax and O^T += V^T P^T of tile j,
  // rebuilds K tile j+2 and V tile j+1 into the free buffers and refills the registers with K
  // tile j+3 and V tile j+2; one barrier ends it.
  constexpr int N_QK = 2 * NKS, N_PV = 4 * NDB, N_MFMA = N_QK + N_PV;
  // operand fragment n from LDS, shared by the wave's row blocks: fragments 0..N_QK-1 are rows of K
  // (32-key block mb = n / NKS), the rest columns of V (k-step kk covers keys 16kk .. 16kk+15 of the
  // tile in the slot order the S^T accumulator already has: slot (g, j) = key 16kk + 8(j/4) + 4g + j%4)
  auto load_frag = [&](auto n_c, const uint16_t* ks, const uint16_t* vs) __attribute__((always_inline)) -> bf16x8 {
    constexpr int n = decltype(n_c)::value;
    if constexpr (n < N_QK) {
      constexpr int mb = n / NKS, kk = n % NKS;
      return *reinterpret_cast<const bf16x8*>(ks + (32 * mb + i) * KS + 16 * kk + 8 * g);
    } else {
      constexpr int m = n - N_QK, kk = m / NDB, db = m % NDB;
      const uint16_t* vrow = vs + (16 * kk + 4 * g + (lp >> 2)) * VS + 16 * dhalf + 4 * (lp & 3);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(vrow + 32 * db));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(vrow + 8 * VS + 32 * db));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  // the MFMA of fragment n for row block r
  auto mfma_with = [&](auto n_c, auto r_c, const bf16x8& f) __attribute__((always_inline)) {
    constexpr int n = decltype(n_c)::value, r = decltype(r_c)::value;
    if constexpr (n < N_QK) {
      constexpr int mb = n / NKS, kk = n % NKS;
      if constexpr (kk == 0) s[r][mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, qf[r][kk], nmref[r], 0, 0, 0);
      else s[r][mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, qf[r][kk], s[r][mb], 0, 0, 0);
    } else {
      constexpr int m = n - N_QK, kk = m / NDB, db = m % NDB;
      o[r][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, pf_get(r_c, IC<kk>{}), o[r][db], 0, 0, 0);
    }
  };
  // ---- plain iteration: first tile, masked tiles, tiles a row block skips, last tile.
  // `mask_c` = the row blocks of this wave that take part (bit r); `part_c` = 0: the whole tile, 1: its
  // logits only (they stay in s), 2: the rest of a tile whose logits are in s already, 3: the logits of
  // its first 32 keys only, 4: the rest of a tile whose first 32 logits are in s already.
  auto cold_compute = [&](int j, auto mask_c, auto part_c) __attribute__((always_inline)) {
    constexpr int M = decltype(mask_c)::value, PART = decltype(part_c)::value;
    const uint16_t* ks = lds_k(j % 3);
    const uint16_t* vs = lds_v(j & 1);
    // operands are read three fragments ahead here too (the V fragments of the first O^T steps
    // while the softmax runs); not with the any-rank loader, whose kernel got slower with it
    constexpr int LA = LOADER == LOAD_TPA_ANY ? 0 : 3;
    bf16x8 fr[N_MFMA];
    // fragments this call uses (0 .. N_QK - 1: K rows, the first NKS of them those of keys 0-31), and which of
    // them belong to the logits
    constexpr int FIRST = PART == 2 ? N_QK : PART == 4 ? NKS : 0, END = PART == 1 ? N_QK : PART == 3 ? NKS : N_MFMA;
    constexpr int QK_END = PART == 3 ? NKS : N_QK;
    static_for<LA>([&](auto n_c) __attribute__((always_inline)) {
      constexpr int n = FIRST + decltype(n_c)::value;
      if constexpr (n < END) fr[n] = load_frag(IC<n>{}, ks, vs);
    });
    if constexpr (PART != 2) {
      static_for<QK_END - FIRST>([&](auto n_c) __attribute__((always_inline)) {
        constexpr int n = FIRST + decltype(n_c)::value;
        if constexpr (n + LA < END) fr[n + LA] = load_frag(IC<n + LA>{}, ks, vs);
        static_for<RB>([&](auto r_c) __attribute__((always_inline)) {
          if constexpr ((M >> decltype(r_c)::value) & 1) mfma_with(IC<n>{}, r_c, fr[n]);
        });
      });
    }
    if constexpr (PART != 1 && PART != 3) {
      static_for<RB>([&](auto r_c) __attribute__((always_inline)) {
        if constexpr ((M >> decltype(r_c)::value) & 1) do_softmax(j, r_c);
      });
      static_for<N_PV>([&](auto n_c) __attribute__((always_inline)) {
        constexpr int n = N_QK + decltype(n_c)::value;
        if constexpr (n + LA < END) fr[n + LA] = load_frag(IC<n + LA>{}, ks, vs);
        static_for<RB>([&](auto r_c) __attribute__((always_inline)) {
          if constexpr ((M >> decltype(r_c)::value) & 1) mfma_with(IC<n>{}, r_c, fr[n]);
        });
      });
    }
  };
  // the loader's share of iteration j: K tile j+2 and V tile j+1 into LDS, K tile j+3 and V tile j+2 on their way
  auto advance_tiles = [&](int j) __attribute__((always_inline)) {
    const uint16_t* a_slot = LOADER == LOAD_TPA_R2 ? lds_a(j & 1) : nullptr;
    if (j + 2 < ntiles) {
      uint32_t aa_k[NPASS];
      fetch_aa(IsK{}, j + 2, a_slot, aa_k);
      commit(IsK{}, j + 2, aa_k);
      issue(IsK{}, min(j + 3, last));
    }
    if (j + 1 < ntiles) {
      uint32_t aa_v[NPASS];
      fetch_aa(IsV{}, j + 1, a_slot, aa_v);
      commit(IsV{}, j + 1, aa_v);
      issue(IsV{}, min(j + 2, last));
    }
  };
  auto cold_iteration = [&](int j) __attribute__((always_inline)) {
    if (j <= wave_last_tile[0]) {
      // where the rows share one id and its keys form one run, only tile 0 can hold keys of another segment (the run's
      // end is the end of the keys this workgroup visits)
      const int ids = has_seg && !(seg_pure && j > 0) ? ids_of_wave.look(lds_seg(j & 1), l) : kAllOfThem;
      masked_ids = ids == kSomeOfThem;
      if (ids != kNoneOfThem) cold_compute(j, IC<1>{}, IC<0>{});
    }
    advance_tiles(j);
  };

  // ---- prologue: K tiles 0 and 1 and V tile 0 into LDS (head factors straight from global memory),
  // the head factors of K tile 2 / V tile 1 in slot 0, those of K tile 3 / V tile 2 pending, the B
  // factors of K tile 2 and V tile 1 in registers
  {
    u32x4 kreg1[NPASS][2];  // K tile 1, on its way during the Q build like tile 0
    issue(IsK{}, 0);
    issue(IsV{}, 0);
    issue_into(kreg1, IsK{}, min(1, last));
    issue_a(min(2, last), min(1, last));
    build_q();
    uint32_t aa0[NPASS], aa1[NPASS], aa2[NPASS];
    fetch_aa(IsK{}, 0, nullptr, aa0);
    fetch_aa(IsV{}, 0, nullptr, aa1);
    commit(IsK{}, 0, aa0);
    commit(IsV{}, 0, aa1);
    if (last >= 1) {
      fetch_aa(IsK{}, 1, nullptr, aa2);
      commit_from(kreg1, IsK{}, 1, aa2);
    }
  }
  issue(IsK{}, min(2, last));
  issue(IsV{}, min(1, last));
  store_a(0);
  issue_a(min(3, last), min(2, last));
  issue_seg(0);
  store_seg(0);
  issue_seg(min(1, last));
  lds_barrier();

  // Per wave: tile 0 plain, then the run of unmasked tiles in the pipelined loop, then plain again (masked
  // tiles, tiles past this wave's causal range, the last tile).  Three separate loops rather than
  // a branch inside one: every wave passes the same number of barriers either way.
  auto tail = [&](int j) __attribute__((always_inline)) {
    // head factors: publish those of K tile j+3 / V tile j+2, fetch those of K tile j+4 / V tile j+3
    store_a((j + 1) & 1);
    issue_a(min(j + 4, last), min(j + 3, last));
    // key segment ids (one wave): publish those of tile j+1, fetch those of tile j+2
    store_seg((j + 1) & 1);
    issue_seg(min(j + 2, last));
    lds_barrier();
  };
  int hot_end = 1;
  if constexpr (LOADER != LOAD_TPA_ANY) {
    int first_masked = lk_r / kTK;                                   // ragged last tile
    int needed = last;                                               // last tile every row block of the wave needs
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      if (p.causal) first_masked = min(first_masked, max(wrow_r[r] + 1, 0) / kTK);  // first tile with a key past the block's first row
      needed = min(needed, wave_last_tile[r]);
    }
    hot_end = max(1, min(min(ntiles - 1, first_masked), needed + 1));
    // segment masks are applied by the plain iteration only: the pipelined loop runs where no
    // key of another segment can turn up (tile 0, which may start before the run, is plain anyway)
    if constexpr (has_seg) if (!seg_pure) hot_end = 1;
  }
  int j = 0;
  for (; j < 1; ++j) { cold_iteration(j); tail(j); }
  if constexpr (LOADER == LOAD_DENSE) {
    // Unmasked tiles 1 .. hot_end - 1 pipelined: tile j's softmax and O^T run beside the logits of
    // tile j+1 (K is a tile ahead in LDS for this).  The logits of tile 1 are computed here, the
    // loop (generated by gen_prefill_loop.py, which documents the register assignment) then runs
    // iterations 1 .. hot_end - 2 and leaves the logits of tile hot_end - 1, which is finished
    // here.  The state goes in and comes back in operands pinned to the loop's registers.
    if (hot_end >= 3) {
      masked_ids = false;
      cold_compute(1, IC<1>{}, IC<1>{});
      auto cat4 = [](const u32x4& a0, const u32x4& a1, const u32x4& a2, const u32x4& a3) __attribute__((always_inline)) -> f32x16 {
        const u32x8 lo = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
        const u32x8 hi = __builtin_shufflevector(a2, a3, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(f32x16, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15));
      };
      auto qv = [&](int ks) __attribute__((always_inline)) { return __builtin_bit_cast(u32x4, qf[0][ks]); };
      const u32x4 z4 = {0, 0, 0, 0};
      const f32x16 qp0 = cat4(qv(0), qv(1), qv(2), qv(3));
      const f32x16 qp1 = NKS > 4 ? cat4(qv(NKS > 4 ? 4 : 0), qv(NKS > 4 ? 5 : 0), qv(NKS > 4 ? 6 : 0), qv(NKS > 4 ? 7 : 0)) : qp0;
      u32x8 kv_k = __builtin_shufflevector(kreg[0][0], NPASS > 1 ? kreg[NPASS - 1][0] : z4, 0, 1, 2, 3, 4, 5, 6, 7);
      u32x8 kv_v = __builtin_shufflevector(vreg[0][0], NPASS > 1 ? vreg[NPASS - 1][0] : z4, 0, 1, 2, 3, 4, 5, 6, 7);
      // tile 1 is odd: its logits sit in the second set (the first set's contents do not matter: the loop's first
      // matrix instructions overwrite them; handing in the same values saves the registers of a zeroed tuple)
      f32x16 sa0 = s[0][0], sa1 = s[0][1], sb0 = s[0][0], sb1 = s[0][1];
      const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)smem;
      u32x16 st16 = {};
      st16[0] = __float_as_uint(mref[0]); st16[1] = __float_as_uint(lsum[0]);
      st16[2] = lds0 + 2 * (L::k_off(0) + i * KS + 8 * g);                                                   // K fragment rows
      st16[3] = lds0 + 2 * (L::v_off(0) + (4 * g + (lp >> 2)) * VS + 16 * dhalf + 4 * (lp & 3));             // V fragment columns
      st16[4] = lds0 + 2 * (L::k_off(0) + lt * KS + 8 * lc);                                                 // this thread's chunk of a K tile
      st16[5] = lds0 + 2 * (L::v_off(0) + lt * VS + 8 * lc);                                                 // ... of a V tile
      st16[6] = kvoff; st16[7] = vvoff;
      auto uni = [](uint32_t x) __attribute__((always_inline)) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
      u32x16 sc16 = {};
      sc16[0] = 1; sc16[1] = uni(hot_end - 1); sc16[2] = uni(last);
      sc16[3] = uni(kTK * p.kb.stride_l * 2); sc16[4] = uni(kTK * p.vb.stride_l * 2);
      sc16[5] = uni(TPP * p.kb.stride_l * 2); sc16[6] = uni(TPP * p.vb.stride_l * 2);
      sc16[7] = 2 * L::kK * 2; sc16[8] = 0;  // K buffers: iteration 1 reads tile 2 in buffer 2 and writes tile 3 into buffer 0
      auto rsrc_words = [&](const uint16_t* base, int bytes) __attribute__((always_inline)) -> u32x4 {
        const uint64_t a64 = reinterpret_cast<uint64_t>(base);
        return u32x4{uni((uint32_t)a64), uni((uint32_t)(a64 >> 32) & 0xffffu), uni((uint32_t)bytes), (uint32_t)kRsrcFlags};
      };
      const u32x4 kbr = rsrc_words(kb_b, k_rows_bytes), vbr = rsrc_words(vb_b, v_rows_bytes);
      if constexpr (D == 128) {
        asm volatile(
#include "gen/prefill_loop_128_dense.inc"
#include "gen/prefill_loop_128_dense_rare.inc"
            : "+{v[0:15]}"(sa0), "+{v[16:31]}"(sa1), "+{v[32:47]}"(sb0), "+{v[48:63]}"(sb1), "+{v[64:79]}"(nmref[0]),
              "+{v[80:95]}"(o[0][0]), "+{v[96:111]}"(o[0][1]), "+{v[112:127]}"(o[0][NDB > 2 ? 2 : 0]), "+{v[128:143]}"(o[0][NDB > 2 ? 3 : 0]),
              "+{v[176:183]}"(kv_k), "+{v[184:191]}"(kv_v), "+{v[204:219]}"(st16), "+{s[32:47]}"(sc16)
            : "{v[144:159]}"(qp0), "{v[160:175]}"(qp1), "{s[48:51]}"(kbr), "{s[52:55]}"(vbr)
            :
#include "gen/prefill_loop_128_dense_clobbers.inc"
        );
      } else if constexpr (NW == 4) {
        asm volatile(
#include "gen/prefill_loop_64_dense4w.inc"
#include "gen/prefill_loop_64_dense4w_rare.inc"
            : "+{v[0:15]}"(sa0), "+{v[16:31]}"(sa1), "+{v[32:47]}"(sb0), "+{v[48:63]}"(sb1), "+{v[64:79]}"(nmref[0]),
              "+{v[80:95]}"(o[0][0]), "+{v[96:111]}"(o[0][1]),
              "+{v[176:183]}"(kv_k), "+{v[184:191]}"(kv_v), "+{v[204:219]}"(st16), "+{s[32:47]}"(sc16)
            : "{v[144:159]}"(qp0), "{s[48:51]}"(kbr), "{s[52:55]}"(vbr)
            :
#include "gen/prefill_loop_64_dense4w_clobbers.inc"
        );
      } else {
        asm volatile(
#include "gen/prefill_loop_64_dense.inc"
#include "gen/prefill_loop_64_dense_rare.inc"
            : "+{v[0:15]}"(sa0), "+{v[16:31]}"(sa1), "+{v[32:47]}"(sb0), "+{v[48:63]}"(sb1), "+{v[64:79]}"(nmref[0]),
              "+{v[80:95]}"(o[0][0]), "+{v[96:111]}"(o[0][1]),
              "+{v[176:183]}"(kv_k), "+{v[184:191]}"(kv_v), "+{v[204:219]}"(st16), "+{s[32:47]}"(sc16)
            : "{v[144:159]}"(qp0), "{s[48:51]}"(kbr), "{s[52:55]}"(vbr)
            :
#include "gen/prefill_loop_64_dense_clobbers.inc"
        );
      }
      kreg[0][0] = __builtin_shufflevector(kv_k, kv_k, 0, 1, 2, 3);
      vreg[0][0] = __builtin_shufflevector(kv_v, kv_v, 0, 1, 2, 3);
      if constexpr (NPASS > 1) {
        kreg[NPASS - 1][0] = __builtin_shufflevector(kv_k, kv_k, 4, 5, 6, 7);
        vreg[NPASS - 1][0] = __builtin_shufflevector(kv_v, kv_v, 4, 5, 6, 7);
      }
      mref[0] = __uint_as_float(st16[0]); lsum[0] = __uint_as_float(st16[1]);
      j = hot_end - 1;
      const bool odd = j & 1;  // uniform
      s[0][0] = odd ? sb0 : sa0;
      s[0][1] = odd ? sb1 : sa1;
      cold_compute(j, IC<1>{}, IC<2>{});
      advance_tiles(j);
      tail(j);
      ++j;
    }
  } else if constexpr (LOADER == LOAD_TPA_R2) {
    // Unmasked tiles 1 .. hot_end - 1 pipelined in blocks of 32 keys: a block's softmax runs beside the
    // logits of the next block, its O^T beside the rebuild of the tiles ahead.  The logits of the first 32
    // keys of tile 1 are computed here; the loop (generated by gen_prefill_loop.py, which documents the
    // register assignment) runs iterations 1 .. hot_end - 2 - everything advance_tiles() and tail() do
    // included - and leaves the logits of the first 32 keys of tile hot_end - 1, which is finished here.
    if (hot_end >= 3) {
      masked_ids = false;
      cold_compute(1, IC<1>{}, IC<3>{});
      auto cat4 = [](const u32x4& a0, const u32x4& a1, const u32x4& a2, const u32x4& a3) __attribute__((always_inline)) -> u32x16 {
        const u32x8 lo = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
        const u32x8 hi = __builtin_shufflevector(a2, a3, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
      };
      auto qv = [&](int ks) __attribute__((always_inline)) { return __builtin_bit_cast(u32x4, qf[0][ks]); };
      const u32x16 qp0 = cat4(qv(0), qv(1), qv(2), qv(3));
      const u32x16 qp1 = NKS > 4 ? cat4(qv(NKS > 4 ? 4 : 0), qv(NKS > 4 ? 5 : 0), qv(NKS > 4 ? 6 : 0), qv(NKS > 4 ? 7 : 0)) : qp0;
      // rows in flight: (pass, rank) tuples of four registers
      u32x16 kv_k = cat4(kreg[0][0], kreg[0][1], kreg[NPASS - 1][0], kreg[NPASS - 1][1]);
      u32x16 kv_v = cat4(vreg[0][0], vreg[0][1], vreg[NPASS - 1][0], vreg[NPASS - 1][1]);
      f32x16 set0 = s[0][0], set1 = {};
      const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)smem;
      u32x16 st16 = {};
      st16[0] = __float_as_uint(mref[0]); st16[1] = __float_as_uint(lsum[0]);
      st16[2] = lds0 + 2 * (L::k_off(0) + i * KS + 8 * g);                                                   // K fragment rows
      st16[3] = lds0 + 2 * (L::v_off(0) + (4 * g + (lp >> 2)) * VS + 16 * dhalf + 4 * (lp & 3));             // V fragment columns
      st16[4] = lds0 + 2 * (L::k_off(0) + lt * KS + 8 * lc);                                                 // this thread's chunk of a K tile
      st16[5] = lds0 + 2 * (L::v_off(0) + lt * VS + 8 * lc);                                                 // ... of a V tile
      st16[6] = kvoff; st16[7] = vvoff;
      st16[8] = lds0 + 2 * L::a_off(0) + 4 * lt;                                                             // head factor pairs of this thread's tokens
      st16[9] = lds0 + 2 * (L::a_off(0) + a_idx);                                                            // where this thread's head factor goes
      st16[10] = a_mat ? va_voff : ka_voff;
      st16[11] = a_pending;
      auto uni = [](uint32_t x) __attribute__((always_inline)) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
      u32x16 sc16 = {};
      sc16[0] = 1; sc16[1] = uni(hot_end - 1); sc16[2] = uni(last);
      sc16[3] = uni(kTK * p.kb.stride_l * 2); sc16[4] = uni(kTK * p.vb.stride_l * 2);
      sc16[5] = uni(TPP * p.kb.stride_l * 2); sc16[6] = uni(TPP * p.vb.stride_l * 2);
      sc16[7] = 1 * L::kK * 2; sc16[8] = 2 * L::kK * 2; sc16[9] = 0;  // K buffers of tiles 1 and 2, and the one tile 3 goes to
      sc16[10] = uni(p.kb.stride_r * 2); sc16[11] = uni(p.vb.stride_r * 2);
      sc16[12] = uni(kTK * (a_mat ? p.va.stride_l : p.ka.stride_l) * 2);
      sc16[13] = uni(a_mat ? 3 : 4);
      auto rsrc_words = [&](const uint16_t* base, int bytes) __attribute__((always_inline)) -> u32x4 {
        const uint64_t a64 = reinterpret_cast<uint64_t>(base);
        return u32x4{uni((uint32_t)a64), uni((uint32_t)(a64 >> 32) & 0xffffu), uni((uint32_t)bytes), (uint32_t)kRsrcFlags};
      };
      const u32x4 kbr = rsrc_words(kb_b, k_rows_bytes), vbr = rsrc_words(vb_b, v_rows_bytes);
      const u32x4 abr = rsrc_words(a_mat ? va_b : ka_b, a_mat ? va_bytes : ka_bytes);
      if constexpr (D == 128) {
        asm volatile(
#include "gen/prefill_loop_128_r2.inc"
#include "gen/prefill_loop_128_r2_rare.inc"
            : "+{v[0:15]}"(set0), "+{v[16:31]}"(set1), "+{v[32:47]}"(nmref[0]),
              "+{v[48:63]}"(o[0][0]), "+{v[64:79]}"(o[0][1]), "+{v[80:95]}"(o[0][NDB > 2 ? 2 : 0]), "+{v[96:111]}"(o[0][NDB > 2 ? 3 : 0]),
              "+{v[144:159]}"(kv_k), "+{v[160:175]}"(kv_v), "+{v[188:203]}"(st16), "+{s[32:47]}"(sc16)
            : "{v[112:127]}"(qp0), "{v[128:143]}"(qp1), "{s[48:51]}"(kbr), "{s[52:55]}"(vbr), "{s[56:59]}"(abr)
            :
#include "gen/prefill_loop_128_r2_clobbers.inc"
        );
      } else if constexpr (NW == 4) {
        asm volatile(
#include "gen/prefill_loop_64_r24w.inc"
#include "gen/prefill_loop_64_r24w_rare.inc"
            : "+{v[0:15]}"(set0), "+{v[16:31]}"(set1), "+{v[32:47]}"(nmref[0]),
              "+{v[48:63]}"(o[0][0]), "+{v[64:79]}"(o[0][1]),
              "+{v[144:159]}"(kv_k), "+{v[160:175]}"(kv_v), "+{v[188:203]}"(st16), "+{s[32:47]}"(sc16)
            : "{v[112:127]}"(qp0), "{s[48:51]}"(kbr), "{s[52:55]}"(vbr), "{s[56:59]}"(abr)
            :
#include "gen/prefill_loop_64_r24w_clobbers.inc"
        );
      } else {
        u32x8 kv_k8 = __builtin_shufflevector(kv_k, kv_k, 0, 1, 2, 3, 4, 5, 6, 7);
        u32x8 kv_v8 = __builtin_shufflevector(kv_v, kv_v, 0, 1, 2, 3, 4, 5, 6, 7);
        asm volatile(
#include "gen/prefill_loop_64_r2.inc"
#include "gen/prefill_loop_64_r2_rare.inc"
            : "+{v[0:15]}"(set0), "+{v[16:31]}"(set1), "+{v[32:47]}"(nmref[0]),
              "+{v[48:63]}"(o[0][0]), "+{v[64:79]}"(o[0][1]),
              "+{v[144:151]}"(kv_k8), "+{v[160:167]}"(kv_v8), "+{v[188:203]}"(st16), "+{s[32:47]}"(sc16)
            : "{v[112:127]}"(qp0), "{s[48:51]}"(kbr), "{s[52:55]}"(vbr), "{s[56:59]}"(abr)
            :
#include "gen/prefill_loop_64_r2_clobbers.inc"
        );
        kv_k = __builtin_shufflevector(kv_k8, kv_k8, 0, 1, 2, 3, 4, 5, 6, 7, 0, 1, 2, 3, 4, 5, 6, 7);
        kv_v = __builtin_shufflevector(kv_v8, kv_v8, 0, 1, 2, 3, 4, 5, 6, 7, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      kreg[0][0] = __builtin_shufflevector(kv_k, kv_k, 0, 1, 2, 3);
      kreg[0][1] = __builtin_shufflevector(kv_k, kv_k, 4, 5, 6, 7);
      vreg[0][0] = __builtin_shufflevector(kv_v, kv_v, 0, 1, 2, 3);
      vreg[0][1] = __builtin_shufflevector(kv_v, kv_v, 4, 5, 6, 7);
      if constexpr (NPASS > 1) {
        kreg[NPASS - 1][0] = __builtin_shufflevector(kv_k, kv_k, 8, 9, 10, 11);
        kreg[NPASS - 1][1] = __builtin_shufflevector(kv_k, kv_k, 12, 13, 14, 15);
        vreg[NPASS - 1][0] = __builtin_shufflevector(kv_v, kv_v, 8, 9, 10, 11);
        vreg[NPASS - 1][1] = __builtin_shufflevector(kv_v, kv_v, 12, 13, 14, 15);
      }
      mref[0] = __uint_as_float(st16[0]); lsum[0] = __uint_as_float(st16[1]);
      a_pending = st16[11];
      j = hot_end - 1;
      s[0][0] = set0;
      cold_compute(j, IC<1>{}, IC<4>{});
      advance_tiles(j);
      tail(j);
      ++j;
    }
  }
  for (; j < ntiles; ++j) { cold_iteration(j); tail(j); }

  // ---- epilogue: normalise, store O[b, qrow, h, :] and LSE[b, h, qrow]
  // A row block's 32 output rows go through the wave's own slice of LDS (free after the last
  // barrier), so that they leave as whole 16-byte chunks of whole rows instead of 8-byte pieces
  // of 32 rows.  (LDS operations of one wave complete in order: the next row block's writes
  // cannot overtake the reads of this one.)
  static_for<RB>([&](auto r_c) __attribute__((always_inline)) {
    constexpr int r = decltype(r_c)::value;
    const float ltot = halves_sum(lsum[r]);
    if constexpr (SPLIT) {
      if (qrow[r] < p.lq) {
        const int64_t row = (((int64_t)range * p.B + b) * p.lq + qrow[r]) * p.H + h;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int vq = 0; vq < 4; ++vq)
            *reinterpret_cast<f32x4*>(pp.part_o + row * D + 32 * db + 8 * vq + 4 * g) =
                f32x4{o[r][db][4 * vq], o[r][db][4 * vq + 1], o[r][db][4 * vq + 2], o[r][db][4 * vq + 3]};
        if (g == 0) pp.part_ml[row] = float2{seen[r] ? mref[r] : -INFINITY, ltot};
      }
      return;
    }
    const float inv = 1.f / ltot;
    constexpr int OS = D + 8;  // row stride (elements)
    uint16_t* const ot = smem + w * 32 * OS;
    static_assert(NW * 32 * OS * sizeof(uint16_t) <= L::kBytes, "output staging fits");
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        u32x2 pk;
        pk[0] = pack_bf16(o[r][db][4 * vq] * inv, o[r][db][4 * vq + 1] * inv);
        pk[1] = pack_bf16(o[r][db][4 * vq + 2] * inv, o[r][db][4 * vq + 3] * inv);
        *reinterpret_cast<u32x2*>(ot + i * OS + 32 * db + 8 * vq + 4 * g) = pk;
      }
    __builtin_amdgcn_wave_barrier();
    constexpr int CPRO = D / 8, RPI = 64 / CPRO;  // 16-byte chunks per row, rows per store instruction
    const int orow_l = l / CPRO, ochunk = l % CPRO;
#pragma unroll
    for (int n = 0; n < 32 / RPI; ++n) {
      const int rr = n * RPI + orow_l;
      const u32x4 val = *reinterpret_cast<const u32x4*>(ot + rr * OS + 8 * ochunk);
      if (wrow0[r] + rr < p.lq)
        // (the output is not read again: stored around the L2, whose room the K/V tiles of the other workgroups
        // need - c2 -2.5 % against ordinary stores)
        __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(p.o + (((int64_t)b * p.lq + wrow0[r] + rr) * p.H + h) * D + 8 * ochunk));
    }
    __builtin_amdgcn_wave_barrier();
    if (qrow[r] < p.lq && p.lse && g == 0)
      p.lse[((int64_t)b * p.H + h) * p.lq + qrow[r]] = (mref[r] + __builtin_amdgcn_logf(ltot)) * kLn2;
  });
}

// Merges the key ranges of a split launch: o = sum_s 2^(m_s - max m) O_s / sum_s 2^(m_s - max m) l_s, lse = ln of the
// total (the rule of _lse_accum, tpa/tpa.py:228-242).  A thread takes 8 elements of one (row, head); all references are
// whole numbers, so every factor is an exact power of two and the split changes no rounding but that of the fp32 sums.
template <int D>
__global__ __launch_bounds__(256) void prefill_merge_kernel(const float* part_o, const float2* part_ml, uint16_t* o, float* lse, int S, int64_t rows, int lq, int H) {
  constexpr int CPR = D / 8;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x, row = idx / CPR;  // row over (b, query row, h)
  const int cc = (int)(idx % CPR);
  if (row >= rows) return;
  float m = -INFINITY;
  for (int s = 0; s < S; ++s) m = fmaxf(m, part_ml[s * rows + row].x);
  float acc[8] = {}, l = 0.f;
  for (int s = 0; s < S; ++s) {
    const float2 ml = part_ml[s * rows + row];
    if (ml.x == -INFINITY) continue;  // this range held no key of the row: nothing was stored for it
    const float f = __builtin_amdgcn_exp2f(ml.x - m);
    const f32x4* at = reinterpret_cast<const f32x4*>(part_o + (s * rows + row) * D + 8 * cc);
    const f32x4 x0 = at[0], x1 = at[1];
    l += f * ml.y;
#pragma unroll
    for (int e = 0; e < 4; ++e) { acc[e] += f * x0[e]; acc[4 + e] += f * x1[e]; }
  }
  const float inv = 1.f / l;  // no visible key: 0 * inf = NaN, as in tpa/tpa.py:437-439
  u32x4 pk;
#pragma unroll
  for (int j = 0; j < 4; ++j) pk[j] = pack_bf16(acc[2 * j] * inv, acc[2 * j + 1] * inv);
  *reinterpret_cast<u32x4*>(o + row * D + 8 * cc) = pk;
  if (lse && cc == 0) {
    const int h = (int)(row % H);
    const int64_t bi = row / H;
    lse[(bi / lq * H + h) * lq + bi % lq] = (m + __builtin_amdgcn_logf(l)) * kLn2;
  }
}

// (batch, head) pairs of an XCD that run side by side (dense loader): enough of them for about 64 workgroups (two
// rounds of an XCD's 32 compute units, so that the heaviest query blocks of a group start together), as few as that
// allows (so that the workgroups resident together are neighbouring blocks of the same pairs).  Measured, dense
// attention: B = 8, T = 2048, H = 64, D = 64 (64 pairs per XCD, 8 blocks each) 0.654 ms with all pairs side by
// side, 0.601 - 0.603 with 1 to 8; B = 4, T = 4096, H = 16 (8 pairs, 16 blocks) 0.250 with 4 or 8, 0.256 with 2,
// 0.291 with 1 (the last group's heavy blocks start late); T = 32768, H = 32 (4 pairs, 128 blocks) 7.04 with 1, 7.21 with 4.
// The sizes of an XCD's groups differ by one at most: a short last one would start its heavy blocks late and leave compute
// units idle.  With the reconstruction, us, a short last group / these, causal: 72 pairs, T = 2048, D = 64 93 / 73, D = 128 140 /
// 112; 80, T = 2048 94 / 78; 136, T = 1024 68 / 57; not causal 40, T = 4096, D = 128 429 / 343, 72 677 / 588, but 104, T = 2048 (of
// eight and five; seven and six) 248 / 259.  The number of groups is the nearest: with 31 pairs per XCD of 4 blocks, causal, 88 us
// in one group of all, 86 in two.
// Of workgroups of four waves 64 are resident on an XCD, and two rounds are 128.  With groups of 64 under the causal mask the second group
// began when the first one's light blocks ended (D = 64, us, groups of 64 / of 128: 4 x 4096, 16 heads 179 / 167.5; 1 x 8192, 16 heads
// 173.6 / 162; 8 x 1500, 16 heads 70.3 / 67.4; 1 x 3200, 64 heads 126.6 / 110.4; documents of 1000 in 1 x 8192, 16 heads 66.3 / 62.0).  From
// eight rounds on a late group weighs little and fewer pairs side by side share more (8 x 1024, 64 heads 139.7 / 141.9), without a
// mask all blocks are alike (8 x 2048, 64 heads 667 / 677).
inline int dense_pair_groups(int npairs, int nqb, bool four_waves, bool causal) {
  const bool late_blocks_weigh = causal && (int64_t)((npairs + 7) / 8) * nqb < 512;
  const int workgroups = four_waves && late_blocks_weigh ? 128 : 64;
  return pair_groups(npairs, (workgroups + nqb - 1) / nqb);
}

// Four waves and 128 query rows per workgroup, two workgroups on a compute unit, in place of eight and 256 (head size 64; at 128 the
// tiles leave room for one).  The two do not wait for each other's barriers, fit documents, the diagonal and a last block of rows
// more closely and fill more compute units where there are few blocks; both stage (or rebuild) every tile, which is what long runs
// of unmasked tiles lose by.  us, eight waves / four, with the reconstruction where the tiles are dense:
//   Without a mask, or with many cached keys, the two are compared by their rounds of 256 workgroups, a round of four waves as half a round of
//     eight and a tenth (dense tiles, few of them: 2 %) of what they stage twice.  1 x 600, 8 heads 20.5 / 17.5; 3 x 1300, 64 heads 138 /
//     131; 8 x 600, 64 heads 123 / 109; 2 x 2000, 16 heads 50.7 / 59.7; rank 2 fused: 8 x 300, 64 heads 59.3 / 46.7; 1 x 300, 64 heads 15.9 /
//     13.6; 1 x 1000, 64 heads 30.1 / 33.8; 8 x 700, 64 heads 130 / 135; chunks of 300 over 2000, 64 heads 200 / 176, of 512 over 8192 305 / 347
//   Causal: up to about a round and a half of eight waves the longest block decides, and half of it ends sooner: 1 x 2048, 32 heads 48.0 / 41.5;
//     3 x 2300, 8 heads 48.6 / 40.4; 1 x 2304, 32 heads 52.8 / 47.2; 1 x 2816, 32 heads 61.1 / 57.5; rank 2 fused: 1 x 700, 16 heads 21.6 / 18.5; 1 x
//     1800, 32 heads 43.3 / 37.9; 4 x 1024, 16 heads 28.7 / 26.7.  But not where the fused kernel's mapping leaves each XCD one block of all
//     heads, light or heavy, and more of them than compute units: 1 x 1024, 64 heads 30.0 / 33.6; 2 x 512, 64 heads 20.4 / 22.8.
//     Beyond, the tiles that all blocks visit decide, of which blocks of 128 rows have fewer (the diagonal, the last block), with 6 % for staging
//     them twice (rank 2 fused, rebuilding: 13 %): 8 x 1024, 64 heads 148 / 141; 8 x 1500, 16 heads 70.5 / 68.4; 4 x 1600, 64 heads 163 / 146; 1 x
//     3200, 64 heads 117 / 111; but 3 x 2048, 16 heads 49.2 / 51.4; 4 x 2048 56.4 / 57.6; 2 x 4000 87.3 / 91.9; 4 x 4096 166 / 169; 1 x 8192 153 / 163;
//     fused 12 x 768, 32 heads 91.9 / 85.6; 16 x 512, 16 heads 36.7 / 34.7.
//   Segment ids: what the rows hold the host cannot see, and documents are what ids are for.  Causal: 3 x 1777, 16 heads, of 421 tokens 43.4 /
//     38.4; 4 x 2500, 64 heads, of 800 236 / 202; 1 x 8192, 16 heads, of 1000 70.9 / 62.2; 1 x 16 384, 16 heads, of 1000 136 / 113, of 4000 234 / 216;
//     one document in every row loses: 4 x 4096, 16 heads 172.5 / 174.5, 2 x 9000, 8 heads 198 / 194, 1 x 8192, 16 heads 153 / 166, 1 x 16 384
//     549 / 571.  Without a mask 4 x 4096, 16 heads, of 1000 148 / 138, one document 289 / 299; 16 x 512, 16 heads, of 100 43.6 / 40.9, one 44.4 / 46.3; but
//     in one round of eight waves 2 x 2000, 16 heads, of 300 31.1 / 34.1, one 51.7 / 60.4.
inline bool wants_four_waves(const PrefillParams& p, bool dense) {
  const int64_t pairs = (int64_t)p.B * p.H, blocks = (int64_t)p.B * ((p.lq + 127) / 128);
  const int64_t eight = pairs * ((p.lq + 255) / 256), four = p.H * blocks;
  const double staging = dense && p.lk <= 1408 ? 1.02 : 1.1;
  const bool rounds = staging * (double)((four + 255) / 256) < 2.0 * (double)((eight + 255) / 256);
  const bool one_block_per_xcd = !dense && blocks == 8 && p.H > 32;  // pair_of_workgroup
  if (p.kvseg) return p.causal ? !one_block_per_xcd : eight > 256 || rounds;
  if (!p.causal || p.lk >= 2 * (int64_t)p.lq) return rounds;  // masked tiles are a small part of all
  if (p.lq > 8192 || p.lk > 8192 || one_block_per_xcd) return false;
  if (eight <= 352 && p.lk <= (dense ? 4096 : 2048)) return true;
  const int offset = p.coff + (p.causal == TPA_CAUSAL_BOTTOM_RIGHT ? p.lk - p.lq : 0);
  auto tiles = [&](int rows) {  // of all blocks of so many query rows
    int64_t n = 0;
    for (int q0 = 0; q0 < p.lq; q0 += rows) n += (max(0, min(p.lk, q0 + rows + offset)) + kTK - 1) / kTK;
    return (double)n;
  };
  return (dense ? 1.06 : 1.13) * tiles(128) < 2.0 * tiles(256);
}

// Batch entries of different lengths, longest first, where a launch is more than a round of workgroups and a half; in one round there is
// nothing to order, and an XCD that meets every entry has more factors to fetch.  Over a cache of at least twice the rows: with fewer keys a
// causal block's place weighs as much as the length.  us before / now, mean of four sets of lengths from half of the cache on (all equal), rank 2: 9 x
// 512 rows over 8192, 16 heads of 128 (288 workgroups) 327 / 334, 5 x 512, 32 heads (320) 342 / 341, 2 x 1500, 32 heads (384) 355 / 347 (422 / 423),
// 3 x 500 over 4000, 64 heads of 64 (384) 129 / 124 (148 / 151); one set, 512 workgroups and more: 8 x 512 over 8192, 32 heads of 128 458 / 391 (523 /
// 525), 4 x 1024 451 / 405 (506 / 508), 4 x 512, 64 heads of 64 272 / 233 (329 / 326), 8 x 300 over 4000 254 / 226 (282 / 285); rank 4, dense tiles: 16 x
// 300 over 4000, 32 heads of 128 648 / 628 (732 / 734).  Ranges do not count as rounds: 7 x 1000 over 9000, 8 heads of 128, 224 blocks in two
// each 241 / 249.  Dense tiles of an XCD belong to a head of every entry anyway; they gain with up to two blocks of rows, and with four 8 x 1024
// over 4096, 32 heads of 128 take 470 / 474 (551 / 564).
// The order costs every workgroup the lengths and their comparison before its first load, which short walks do not get back, nor those of many
// entries, whose lengths level out by themselves: 44 x 47 rows over 113, 16 heads of 64, rank 4 24.9 / 34.4; 48 x 27 over 200, 64 heads 72 / 88; 25 x 103 over 406, 32
// heads of 128 87 / 95; 40 x 633 over 1808, 8 heads of 64 106 / 122; 33 x 159 over 2036 96 / 103.  Up to 32 entries over 2048 keys and more: mean of 88 shapes, half to
// all of the cache, 0.95 (fused) and 0.96 (dense) of the time without the order, 0.83 - 1.05; all lengths equal 0.99 and 1.00 (67 shapes, 0.94 - 1.03).  Shorter
// caches 1.015 fused and 0.99 dense, more entries 1.07 and 1.00.  (The grid covers eight groups of heads as well: they are npairs * H workgroups.)
bool longest_first_pays(const PrefillParams& p, bool dense) {
  return p.kvlen && (!dense || p.lq <= 2 * kBQ) && p.B > 1 && p.B <= kMostOrdered && p.H % 8 == 0 && p.lk >= std::max<int64_t>(2048, 2 * (int64_t)p.lq) && (int64_t)p.npairs * p.H >= 384 * p.S;
}

template <int D, int LOADER, bool SEG = false, bool SPLIT = false, int NW = 8, bool ORDER = false>
int launch_prefill(const PrefillParams& p, hipStream_t stream) {
  if constexpr (!SEG && !SPLIT && NW == 8 && !ORDER)
    if (p.S > 1) return launch_prefill<D, LOADER, SEG, true>(p, stream);
  PrefillParams q = p;
  if constexpr (D == 64 && LOADER != LOAD_TPA_ANY && !SPLIT && NW == 8 && !ORDER) {
    if (wants_four_waves(p, LOADER == LOAD_DENSE)) {
      q.nqb = (p.lq + kBQ / 2 - 1) / (kBQ / 2);
      q.npairs = q.nqb * p.B;
      return launch_prefill<D, LOADER, SEG, SPLIT, 4>(q, stream);
    }
  }
  if constexpr (!SEG && !ORDER)
    if (longest_first_pays(p, LOADER == LOAD_DENSE)) return launch_prefill<D, LOADER, SEG, SPLIT, NW, true>(p, stream);
  auto kern = prefill_kernel<D, LOADER, SEG, SPLIT, NW, ORDER>;
  constexpr size_t lds_bytes = Lds<D>::kBytes;
  static bool configured[kMaxDevices] = {};
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), lds_bytes); rc != TPA_OK) return rc;
  // one workgroup per (query block, batch, head): see the kernel for how ids map to them
  int64_t n;
  if (LOADER == LOAD_DENSE) {
    q.pair_groups = dense_pair_groups(p.B * p.H, p.nqb, NW == 4, p.causal != 0);
    n = pair_group_workgroups(p.B * p.H, p.nqb);
  } else {
    q.head_groups = head_groups(p.npairs, p.H);
    n = workgroups_of(p.npairs, p.H, q.head_groups);
  }
  if (n > 2147483647LL) return TPA_ERR_SHAPE;
  dim3 grid((unsigned)n);
  hipLaunchKernelGGL(kern, grid, dim3(NW * 64), lds_bytes, stream, q);
  if constexpr (SPLIT) {
    if (hipGetLastError() != hipSuccess) return TPA_ERR_LAUNCH;
    const int64_t rows = (int64_t)p.B * p.lq * p.H;
    hipLaunchKernelGGL((prefill_merge_kernel<D>), dim3((unsigned)((rows * (D / 8) + 255) / 256)), dim3(256), 0, stream, p.part_o, p.part_ml, p.o, p.lse, p.S, rows, p.lq, p.H);
  }
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

// Key ranges per query block.  Without them a launch of fewer workgroups than compute units takes as long as the block
// with the most tiles; with them the partial results make a trip through memory and every workgroup pays its prologue
// again.  The choice minimises an estimate in us: 1.7 per tile (D = 128; 1.3 at D = 64), 7 per workgroup, 7 for the merge
// and the partial results at 4 TB/s; the launch takes its rounds of 256 average workgroups, or the heaviest workgroup.
// Measured, us without / with ranges: a chunk of 331 tokens over 2258 keys, 16 heads of 128: 97 / 73; 608 over 11433, 8
// heads of 64: 182 / 76; one sequence of 4096 tokens, 8 heads of 64, causal: 70 / 47.
// Fewer than 24 tiles: of 2 and more blocks 512 to 1400 rows gain at most 8 % and lose up to twofold.  One block, where the ranges
// find compute units that have nothing to do: a tile of the rank-2 rebuild is 2.0 us (1.1 at D = 64), one of dense arrays 1.75 in rank 2 (110 shapes of 380 to 768 keys,
// 1.066 of one range's speed, 1.10 with the best count for each), of other ranks 1.55 (0.65),
// a second range 9.5 and its partial results.  140 rows over 1160 keys, us without / with: rank 2, 8 heads of 128 44.4 / 29.6, 2 x 32 heads of 128
// 45.1 / 39.5, 8 heads of 64 25.7 / 21.9; rank 4, 8 heads of 128 35.6 / 26.7; 4 x 16 heads of 64 26.2 / 26.2 (one range), rank 4 29.7 / 31.3 (one).
// (What counts there is the `reach` of the mask, not the length of the cache: 33 rows over 861 keys from the first one on, 2 x 16 heads of 64, rank 2:
// eight ranges, all but one empty, 11.7, one 6.7.  And the tiles of the route: 217 over 437, 4 x 8 heads of 128, dense 23.7, in two ranges 28.9; 85 over 612, 2 x 8 24.2, in
// five 22.8.)
int choose_splits(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D, int64_t rk, bool causal, int64_t reach, bool dense) {
  const int64_t blocks = (lq + kBQ - 1) / kBQ, wgs = blocks * B * H;
  const double per_tile = D == 128 ? 1.7 : 1.3, per_wg = 7.0, most = (double)((lk + kTK - 1) / kTK);
  // tiles of an average block: under the causal mask the first one sees (lk - lq + 256) keys, the last one all
  const double least = lk > lq ? (double)(lk - lq) / kTK : 0.0, avg = causal ? 0.5 * (least + most) + 2.0 : most;
  int best = 1;
  if (most < 24) {  // a block's own tiles take 40 us at most: little to win over the merge, but where one block has them all
    if (blocks > 1) return 1;
    const double tile = rk == 2 ? (D == 128 ? (dense ? 1.75 : 2.0) : 1.1) : (D == 128 ? 1.55 : 0.65);
    const int64_t tiles = (reach + kTK - 1) / kTK;
    double gain = 1.5;
    for (int S = 2; S <= 8 && wgs * S <= 256; ++S) {
      const double us = tile * (double)(tiles - (tiles + S - 1) / S) - 9.5 - (double)S * B * lq * H * D * 8.0 / 4e6;
      if (us > gain) { best = S; gain = us; }
    }
    return best;
  }
  double best_us = 0.0;
  for (int S = 1; S <= 16 && wgs * S <= 1024 && (S == 1 || most >= 2 * S); ++S) {
    const double heaviest = per_wg + per_tile * (double)(((int64_t)most + S - 1) / S), all = (double)((wgs * S + 255) / 256) * (per_wg + per_tile * avg / S);
    const double us = (heaviest > all ? heaviest : all) + (S > 1 ? 7.0 + (double)S * B * lq * H * D * 8.0 / 4e6 : 0.0);
    if (S == 1 || us < (best == 1 ? 0.92 : 1.0) * best_us) { best = S; best_us = us; }
  }
  return best;
}
size_t split_bytes(int64_t B, int64_t lq, int64_t H, int64_t D, int64_t S) { return S > 1 ? (size_t)(S * B * lq * H * (D + 2) * 4) : 0; }

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }
bool factor_ok(const TpaFactor& f) {
  return aligned16(f.ptr) && f.stride_b % 8 == 0 && f.stride_l % 8 == 0 && f.stride_r % 8 == 0;
}
// one batch entry of a K/V-side array is addressed through a buffer resource with 32-bit byte
// offsets: its extent must stay below 2 GiB and its strides must not be negative
bool range_ok(const TpaFactor& f, int64_t tokens, int64_t ranks, int64_t width) {
  if (f.stride_l < 0 || f.stride_r < 0) return false;
  return ((tokens - 1) * f.stride_l + (ranks - 1) * f.stride_r + width) * 2 < (int64_t(1) << 31);
}

}  // namespace
}  // namespace tpa


int tpa_prefill_mfma_supported(const TpaFwdArgs* a) {
  if (a->dtype != TPA_DTYPE_BF16) return 0;
  if (a->dk != a->dv || (a->dk != 64 && a->dk != 128)) return 0;
  if (!(a->sm_scale > 0.f)) return 0;
  if (!tpa::factor_ok(a->qb) || !tpa::factor_ok(a->kb) || !tpa::factor_ok(a->vb)) return 0;
  if (!tpa::range_ok(a->kb, a->lk, a->rk, a->dk) || !tpa::range_ok(a->vb, a->lk, a->rk, a->dv) ||
      !tpa::range_ok(a->ka, a->lk, a->rk, 1) || !tpa::range_ok(a->va, a->lk, a->rk, 1))
    return 0;
  if (!tpa::aligned16(a->o)) return 0;
  return 1;
}

// bytes of workspace that let the prefill kernel run on dense Q [B, lq, H, D], K and V [B, lk, H, D]
// (bf16, each rounded up to 256 bytes); 0 if a batch entry would not fit the kernel's 32-bit tile offsets
size_t tpa_prefill_dense_bytes(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D) {
  if (lk * H * D * 2 >= (int64_t(1) << 31)) return 0;
  const auto slot = [](int64_t n) { return (size_t)((n * 2 + 255) / 256 * 256); };
  return slot(B * lq * H * D) + 2 * slot(B * lk * H * D);
}

// Whether reconstructing dense Q, K and V once (one HBM-bound launch) and running the plain tile
// loader beats rebuilding every tile in the flash loop, by the lengths and the rank alone.  The loop over dense tiles overlaps the
// logits of one tile with the softmax of the one before and has no rebuild in it; the
// reconstruction grows with the length only.  Rank 2 has a tuned rebuild in the fused kernel:
// measured at B * H = 64, D = 128 the two routes meet at 1024 rows (51 against 52 us) and the dense
// one wins from 2048 on (105 against 115 us; 4096: 0.32 against 0.38 ms).  Other ranks loop over
// the ranks per tile in the fused kernel: dense from the second query block on.
// One query block rebuilds every tile once on either route, so there the rebuild itself decides.  Fused over dense time
// at 17 to 256 rows over 1024 to 16384 keys, 1 to 8 sequences of 8 to 64 heads of 64 and 128, keys split where that pays:
// rank 1 0.65 - 1.37 (over 1 only up to 1024 keys and for small batches of up to 4096; 8 sequences of 32 heads over 4096 keys
// 170 against 253 us), rank 3 0.94 - 1.8, rank 4 0.99 - 2.0, rank 8 1.25 - 5.5, rank 16 1.4 - 9.5.  So from rank 3 on
// dense, which takes 4 lk H D bytes per sequence for K and V where the fused kernel takes none.
int tpa_prefill_wants_dense(int64_t lq, int64_t lk, int64_t rk) {
  if (rk == 2) return lq >= 2048;
  return lq > tpa::kBQ || (rk > 2 && lq > 16 && lk >= 1024);
}

namespace tpa {
namespace {
// One block of query rows over fewer than 1024 keys, any rank but 2: the rebuild that the fused kernel does for every tile of 64 keys,
// against a launch more and the trip of the dense arrays through memory.  Fitted to 500 shapes of 17 to 256 rows, 8 to 1024 (batch,
// head) pairs, ranks 1, 3, 4 and 8 (us, within 5 of each): a tile costs 0.55 + 0.36 R more where it is rebuilt at head size 64, 0.55 + 0.57 R
// at 128 (there rank 8 more than that, its loop waits for every rank's loads), for every round of workgroups a compute unit takes - at 64 two of them share
// one, so that pairs beyond 256 add 0.7 of a round.  Fused / dense, us: rank 4, 1 x 250 rows, 8 heads of 64 17.3 / 12.1; 2 x 130 over 900, 32 heads of 128
// 73.7 / 42.1; 12 x 200, 32 heads of 128 57.8 / 42.9; 8 x 200, 64 heads of 64 27.7 / 34.3 (stays fused); 4 x 40, 64 heads of 64 9.6 / 10.8 (stays);
// rank 8, 1 x 130 over 900, 16 heads of 128 188 / 34; rank 1, 1 x 130 over 900, 8 heads of 64 31.2 / 20.2; 8 x 250, 32 heads of 128 22.6 / 32.2 (stays).
bool one_block_pays(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D, int64_t rk) {
  if (lk >= 1024 || H % 8 != 0) return false;  // beyond that the rule above has spoken; other head counts take three launches
  const double pairs = (double)(B * H), tiles = (double)((lk + kTK - 1) / kTK), mb = pairs * (double)((lq + 2 * lk) * D) * 2e-6;
  if (D == 64) return (pairs > 366 ? pairs / 366 : 1.0) * tiles * (0.55 + 0.36 * rk) > 4.5 + 0.28 * mb;
  return (double)((B * H + 255) / 256) * tiles * (0.55 + 0.57 * rk) > 2.0 + 0.21 * mb;
}
// The same for one call, whose mask and ranks of Q are known, in us.  What the mask hides is neither made dense nor met, and a block of documents, whose lengths
// the host does not know, meets between as many keys as it has rows, with two tiles, and all: half way; the fused kernel sums Q rank by rank, which the dense launch does in passing.  Fitted to 1400 shapes of 17 to 256
// rows, ranks 1 to 8 (1, 2, 4, 6, 16 of Q), within 1.1 us for the half of them.  The line above alone took 48 of 917 to the slower side by more than 2 %,
// with this 15, at the same gain over all (1.24).  Fused / dense: 47 rows over 882 keys from the first one on, 11 x 16 heads of 128, ranks 2, 3 10.4 / 14.1; 95 over
// 867 in documents of 100, 4 x 64 heads of 64, 2, 3 11.8 / 20.9; 227 x 227, 2 x 32 of 128, 2, 1 14.6 / 18.3; 102 x 172, 9 x 16, 2, 3 18.4 / 21.5 (all stay
// fused); 59 over 127 from the first on, 2 x 32 of 128, 16, 3 24.1 / 12.8; 79 x 79, 4 x 8, 4, 3 15.5 / 12.0.
double one_block_saves_us(const TpaFwdArgs* a) {
  const int64_t pairs = (int64_t)a->B * a->H, made = keys_in_reach(a);
  if (!made) return 0.0;  // the rows end before Q is needed
  const int64_t met = a->kv_segment_ids ? (made + std::min<int64_t>(made, a->lq + 2 * kTK)) / 2 : made, tiles = (met + kTK - 1) / kTK;
  const double mb = (double)(pairs * (a->lq + 2 * made) * a->dk) * 2e-6;
  if (a->dk == 64) {
    const double rounds = pairs > 366 ? (double)pairs / 366 : 1.0;
    return rounds * ((double)tiles * (0.21 + 0.30 * a->rk) + 0.41 * a->rq) - 2.9 - 0.13 * mb;
  }
  return (double)((pairs + 255) / 256) * ((double)tiles * (0.12 + 0.54 * a->rk) + 0.86 * a->rq) - 3.5 - 0.22 * mb;
}
// Rank 2 at head size 128: the fused kernel's Q, summed rank by rank through LDS, takes longer than the launch that makes dense arrays, as long as
// these are few.  us, fused / dense, rank 6 of Q, by (batch, head) pairs: 8, 64 rows over 64 keys 14.2 / 10.4, 200 x 600 25.9 / 22.9; 32, 200 x 200 20.6 /
// 17.7, 200 x 600 31.1 / 28.8, 40 x 900 26.9 / 28.8; 64, 130 x 130 18.6 / 16.6, 250 x 250 21.1 / 21.2; 128, 64 x 64 14.4 / 13.1, 130 x 130 18.7 / 19.5.
// (16, 250 x 1000 31.8 / 31.7: from twelve tiles on the walk counts, not Q.  Head size 64: 0.82 - 1.15 with no such line.)
constexpr int kSlowQ = 6;  // ranks of Q from which that holds
bool one_block_of_rank_2_pays(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D) {
  return D == 128 && H % 8 == 0 && lq <= kBQ && lk <= 12 * kTK && B * H * (lq + 2 * lk) <= 40000;
}
// The same for one call, of which the number of workgroups (of 256 rows) is known.  Rank 2 below 2048 rows, dense over fused time, no
// mask / causal / packed documents, 8 to 400 (batch, head) pairs of 512 to 2040 rows each (head size 64 with four or eight waves as
// wants_four_waves has it for either):
//   at most 64 workgroups: the prologue with its loads and Q is most of the time, and shorter without the factors.  D = 128
//     0.78 - 0.86 (8 pairs of 512 rows 27.4 / 22.5 us); D = 64 0.87 - 0.99, with more keys than rows up to 1.16, not taken
//   65 to 256: every compute unit rebuilds for itself and the reconstruction is a launch more.  D = 64 0.92 - 1.32 (128 pairs of 512
//     rows 19.5 / 25.8, but 24 pairs of 2040 40.1 / 37.0), D = 128 0.84 - 1.10 (128 pairs of 512 31.5 / 34.5, but 24 of 2040 66.7 / 58.3)
//   more, from 1000 rows on: D = 64 0.83 - 0.98 (48 pairs of 1777 49.1 / 43.1, with documents of 421 tokens 39.3 / 38.2), D = 128 0.77 - 0.99
//   more, of fewer rows: 512 rows 1.01 - 1.07, 700 to 900 0.81 - 0.99, with more keys than rows up to 1.32
bool dense_pays(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D, int64_t rk) {
  if (tpa_prefill_wants_dense(lq, lk, rk)) return true;
  if (rk != 2) return one_block_pays(B, lq, lk, H, D, rk);
  if (lq <= kBQ) return one_block_of_rank_2_pays(B, lq, lk, H, D);
  if (lk > 5 * lq) return false;
  const int64_t wgs = B * H * ((lq + kBQ - 1) / kBQ);
  return wgs <= 64 ? D == 128 : wgs > 256 && lq >= 1000;
}
}  // namespace
}  // namespace tpa

size_t tpa_prefill_best_bytes(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D, int64_t rk) {
  const size_t dense = tpa::dense_pays(B, lq, lk, H, D, rk) ? tpa_prefill_dense_bytes(B, lq, lk, H, D) : 0;
  const int s0 = tpa::choose_splits(B, lq, lk, H, D, rk, false, lk, false), s1 = tpa::choose_splits(B, lq, lk, H, D, rk, true, lk, false);
  return dense + tpa::split_bytes(B, lq, H, D, s0 > s1 ? s0 : s1);
}

namespace tpa {
namespace {

// What a call wants of a workspace: dense Q, K and V (0: the fused kernel), and behind them the partial results of S key
// ranges per query block (the kernels with segment ids do not split the keys).
struct PrefillRoute {
  size_t dense;
  int S;
};
// One block of rows is made dense for the time of one launch, so only where the factors allow that and this very call saves by it.
bool one_block_of_call_pays(const TpaFwdArgs* a) {
  return tpa_recon_dense_qkv_takes(a) && (a->rk == 2 ? a->rq >= kSlowQ : one_block_saves_us(a) > 0.5);
}
int splits_of_call(const TpaFwdArgs* a, bool dense) {
  if (a->kv_segment_ids) return 1;
  const int tiles = (int)(((int64_t)a->lk + kTK - 1) / kTK);  // a caller's count beyond that only adds empty ranges
  if (a->num_splits > 0) return std::min(a->num_splits, tiles);
  const bool causal = a->causal != 0;
  return std::min(choose_splits(a->B, a->lq, a->lk, a->H, a->dk, a->rk, causal, a->lk, false),  // of which the room by sizes alone takes account
                  choose_splits(a->B, a->lq, a->lk, a->H, a->dk, a->rk, causal, keys_in_reach(a), dense));
}
PrefillRoute route_of(const TpaFwdArgs* a) {
  const bool pays = dense_pays(a->B, a->lq, a->lk, a->H, a->dk, a->rk) &&
                    (tpa_prefill_wants_dense(a->lq, a->lk, a->rk) || (a->rk == 2 && a->lq > kBQ) || one_block_of_call_pays(a));
  const size_t dense = pays ? tpa_prefill_dense_bytes(a->B, a->lq, a->lk, a->H, a->dk) : 0;
  return {dense, splits_of_call(a, dense != 0)};
}

}  // namespace
}  // namespace tpa

size_t tpa_prefill_call_bytes(const TpaFwdArgs* a) {
  const tpa::PrefillRoute route = tpa::route_of(a);
  return route.dense + tpa::split_bytes(a->B, a->lq, a->H, a->dk, route.S);
}

int tpa_prefill_mfma_launch(const TpaFwdArgs* a, hipStream_t stream) {
  using namespace tpa;
  PrefillParams p{};
  p.qa = a->qa; p.qb = a->qb; p.ka = a->ka; p.kb = a->kb; p.va = a->va; p.vb = a->vb;
  p.qseg = a->q_segment_ids; p.kvseg = a->kv_segment_ids; p.kvlen = a->kv_lengths;
  p.o = static_cast<uint16_t*>(a->o); p.lse = a->lse;
  p.B = a->B; p.lq = a->lq; p.lk = a->lk; p.H = a->H; p.rq = a->rq; p.rk = a->rk;
  p.sm_scale = a->sm_scale; p.causal = a->causal; p.coff = tpa::causal_offset_of(a);
  p.nqb = (a->lq + kBQ - 1) / kBQ;
  p.npairs = p.nqb * a->B;
  // With a workspace Q (times sm_scale * log2 e), K and V are reconstructed once as dense bf16 and
  // the kernel runs with its plain tile loader: no workgroup rebuilds tiles from the rank factors
  // (the fused kernel does that once per workgroup's query rows and head).
  const bool usable = a->workspace && !(reinterpret_cast<uintptr_t>(a->workspace) & 255);
  const PrefillRoute route = route_of(a);
  const bool dense = usable && route.dense && a->workspace_bytes >= route.dense;
  // what the workspace has beyond that can take the partial results of key ranges
  p.S = 1;
  const size_t used = dense ? route.dense : 0;
  const int S = route.S;
  if (usable && S > 1 && a->workspace_bytes >= used + split_bytes(a->B, a->lq, a->H, a->dk, S)) {
    p.S = S;
    p.part_o = reinterpret_cast<float*>(static_cast<char*>(a->workspace) + used);
    p.part_ml = reinterpret_cast<float2*>(p.part_o + (size_t)S * a->B * a->lq * a->H * a->dk);
    p.nqb *= S;
    p.npairs *= S;
  }
  if (dense) {
    const int64_t hd = (int64_t)a->H * a->dk;
    const size_t kv_slot = ((size_t)a->B * a->lk * hd * 2 + 255) / 256 * 256;
    uint16_t* kd = static_cast<uint16_t*>(a->workspace);
    uint16_t* vd = kd + kv_slot / 2;
    uint16_t* qd = vd + kv_slot / 2;
    WindowJob windows{};
    const bool ahead = p.kvseg && windows_ahead_pay(a->B, a->H, a->lq, a->lk, a->rk >= 16 ? 0 : 4096);
    if (ahead) {
      const int rows = a->dk == 64 && wants_four_waves(p, true) ? kBQ / 2 : kBQ;  // as launch_prefill has it
      windows = WindowJob{p.qseg, p.kvseg, p.kvlen, a->lq, a->lk, rows, 0, a->causal, p.coff, reinterpret_cast<int32_t*>(p.o),
                          a->lq * hd / 2, rows * hd / 2, a->dk / 2, a->H};
    }
    int rc = tpa_recon_dense_qkv_bf16(a, qd, kd, vd, a->sm_scale * kLog2e, windows, stream);
    p.windows = ahead && rc == TPA_OK;
    if (rc == TPA_ERR_UNSUPPORTED) {
      rc = tpa_recon_dense_bf16(&a->ka, &a->kb, kd, a->B, a->lk, a->H, a->dk, a->rk, 1.f, stream);
      if (rc == TPA_OK) rc = tpa_recon_dense_bf16(&a->va, &a->vb, vd, a->B, a->lk, a->H, a->dv, a->rk, 1.f, stream);
      if (rc == TPA_OK) rc = tpa_recon_dense_bf16(&a->qa, &a->qb, qd, a->B, a->lq, a->H, a->dk, a->rq, a->sm_scale * kLog2e, stream);
    }
    if (rc != TPA_OK) return rc;
    p.qb = TpaFactor{qd, a->lq * hd, hd, 0};
    p.kb = TpaFactor{kd, a->lk * hd, hd, 0};
    p.vb = TpaFactor{vd, a->lk * hd, hd, 0};
    p.q_scaled = 1;
    if (p.kvseg) {
      if (a->dk == 128) return launch_prefill<128, LOAD_DENSE, true>(p, stream);
      return launch_prefill<64, LOAD_DENSE, true>(p, stream);
    }
    if (a->dk == 128) return launch_prefill<128, LOAD_DENSE>(p, stream);
    return launch_prefill<64, LOAD_DENSE>(p, stream);
  }
  if (p.kvseg) {
    if (a->dk == 128) {
      if (a->rk == 2) return launch_prefill<128, LOAD_TPA_R2, true>(p, stream);
      return launch_prefill<128, LOAD_TPA_ANY, true>(p, stream);
    }
    if (a->rk == 2) return launch_prefill<64, LOAD_TPA_R2, true>(p, stream);
    return launch_prefill<64, LOAD_TPA_ANY, true>(p, stream);
  }
  if (a->dk == 128) {
    if (a->rk == 2) return launch_prefill<128, LOAD_TPA_R2>(p, stream);
    return launch_prefill<128, LOAD_TPA_ANY>(p, stream);
  }
  if (a->rk == 2) return launch_prefill<64, LOAD_TPA_R2>(p, stream);
  return launch_prefill<64, LOAD_TPA_ANY>(p, stream);
}

int mha_prefill_mfma_supported(const MhaFwdArgs* a) {
  if (a->dtype != TPA_DTYPE_BF16) return 0;
  if (a->dk != a->dv || (a->dk != 64 && a->dk != 128)) return 0;
  if (a->bias) return 0;
  if (!(a->sm_scale > 0.f)) return 0;
  if (!tpa::aligned16(a->q) || !tpa::aligned16(a->k) || !tpa::aligned16(a->v) || !tpa::aligned16(a->o)) return 0;
  if ((int64_t)a->lk * a->H * (a->dk > a->dv ? a->dk : a->dv) * 2 >= (int64_t(1) << 31)) return 0;  // 32-bit buffer offsets per batch entry
  return 1;
}

int mha_prefill_mfma_launch(const MhaFwdArgs* a, hipStream_t stream) {
  using namespace tpa;
  PrefillParams p{};
  const int64_t hd = (int64_t)a->H * a->dk;
  p.qb = TpaFactor{a->q, a->lq * hd, hd, 0};
  p.kb = TpaFactor{a->k, a->lk * hd, hd, 0};
  p.vb = TpaFactor{a->v, a->lk * hd, hd, 0};
  p.qa = p.ka = p.va = TpaFactor{nullptr, 0, 0, 0};
  p.o = static_cast<uint16_t*>(a->o); p.lse = a->lse;
  p.B = a->B; p.lq = a->lq; p.lk = a->lk; p.H = a->H; p.rq = 1; p.rk = 1;
  p.sm_scale = a->sm_scale; p.causal = a->causal ? TPA_CAUSAL_TOP_LEFT : TPA_CAUSAL_NONE; p.coff = 0;
  p.nqb = (a->lq + kBQ - 1) / kBQ;
  p.npairs = p.nqb * a->B;
  p.S = 1;
  if (a->dk == 128) return launch_prefill<128, LOAD_DENSE>(p, stream);
  return launch_prefill<64, LOAD_DENSE>(p, stream);
}
