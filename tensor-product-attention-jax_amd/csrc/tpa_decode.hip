// Decode over the factored KV cache for gfx950: a few query tokens against a long cache, split
// over key ranges, built to be bound by HBM bandwidth.
//
// The cache is never expanded to per-head K/V.  With Qm[h, :] = (c / (Rq Rk)) sum_i qa[i, h] qb[i, :]
// the logits are  s[h, t] = sum_j a_k[t, j, h] * (Qm[h, :] . b_k[t, j, :])  and the output is
// o[h, :] = (1/Rk) sum_t sum_j (p[h, t] a_v[t, j, h]) b_v[t, j, :]  (the rank-shared products of
// the non-materialising form, tpa/tpa.py:333-359,398-413), so the rows b_k[(t, j), :] and
// b_v[(t, j), :] are plain row-major matrices that feed two skinny MFMA contractions with the
// heads as the N dimension.  Every cache byte is read from HBM exactly once for all heads.
//
// A workgroup has 4 independent waves; each streams its own range of 32-row blocks
// (32 / Rk tokens) with fully coalesced 16-byte loads that stay in flight in registers two
// blocks ahead, stages the block in its private LDS region (XOR-swizzled so that both the
// 16-byte operand reads and the transposed reads are bank-conflict free), and keeps a private
// online softmax (tpa/tpa.py:389-424).  The waves are merged through LDS, the key ranges
// through a workspace and a small second kernel, both with the rule of _lse_accum
// (tpa/tpa.py:228-242).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "tpa_common.h"

namespace tpa {
namespace {

constexpr int kWaves = 4;
constexpr int kRowsPerBlock = 32;
constexpr int kRsrcFlags = 0x00020000;  // raw 32-bit data format
// How the cache is read: through buffer resources with or without the non-temporal hint, or, where the rows lie too far apart for
// the 32-bit offsets of these (31 rows in a block) or in descending order, with an address per lane.
enum class Reads { kOrdinary, kStreaming, kFar };
constexpr int64_t kFarthestRow = 1 << 25;  // elements between neighbouring rows, at most, for the first two
constexpr int kMinKeys = kWaves * kRowsPerBlock / 2;  // keys of a range with one block of rank 2 per wave
// The same of the call's rank, from rank 4 on
inline int least_keys(int rk) { return rk <= 2 ? kMinKeys : kWaves * kRowsPerBlock / rk; }
// Ranges up to which that counts: beyond, in bf16 at head size 64, the partials of twice the ranges cost more than a second block.  us, by the sizes
// alone / by rank: rank 4, 16 to 63 ranges 1 x 700, 64 heads 8.7 / 8.1, 4 x 1000, 16 heads, two rows 9.7 / 8.6, 2 x 1500, 8 heads 8.6 / 8.3; more 1 x 8000, 32
// heads, two rows 13.3 / 15.2, 1 x 8000, 8 heads 10.5 / 12.0; rank 8, over 127 1 x 7724, 8 heads 12.9 / 13.9, 1 x 8812, two rows 14.7 / 15.7.
inline int most_by_rank(int dtype, int D, int rk) { return dtype == TPA_DTYPE_BF16 && D == 64 && rk <= 8 ? 16 * rk : INT32_MAX; }


struct DecodeParams {
  TpaFactor qa, qb, ka, kb, va, vb;
  float* part_o;  // [range, lq, H, D] fp32, unnormalised; the ranges of a batch entry are neighbours
  float* part_m;  // [range, lq, H] running max (log2 domain)
  float* part_l;  // [range, lq, H] sum of exp2
  const int32_t* kvlen;  // [B] keys per batch entry, or null (= lk)
  const int32_t* page_table;  // paged cache: [B, pages_per_seq] physical page of each logical page
  int page_size, pages_per_seq;  // tokens per page; table row length
  int page_shift;  // log2 of the rows (token, rank) of a page, or -1: no power of two
  int B, lq, lk, H, rq;
  int climit;      // query row qi sees its first qi + climit keys (causal: offset + 1; otherwise lk, no limit)
  int cbr;         // causal, last query aligned with the last key of each batch entry: climit counts from len - lq_total
  int row0;        // this call serves query rows row0 .. row0 + lq - 1 of lq_total (outputs are indexed with them)
  int lq_total;
  int S;           // key ranges per batch entry (slots == 0)
  int slots;       // > 0: the ranges are dealt by the batch entries' lengths, this many at most (plan_ranges)
  float round_keys;  // slots > 0: ranges are this many keys long, or a multiple (a block for each wave); 0: any length
  float min_keys;    // slots > 0: and no shorter than this
  float qscale;    // sm_scale * log2(e) / (rq * rk)
};

// Key ranges dealt by length.  With one count for all batch entries a launch lasts as long as the longest entry takes,
// and shorter ones leave their compute units early; so every entry gets as many ranges as its length asks for at one
// common range length, the shortest one that needs no more than `slots` ranges (one workgroup per compute unit).  The
// lengths are known on the device only, so each wave works the plan out for itself: lane = batch entry (B <= 64) for the
// lengths, lane = candidate range length for the search.  What rounding does to a count only moves the balance: an
// entry's blocks are dealt round-robin to whatever number of ranges it has, at least one.  But the decode kernel and the
// merge each work the plan out and must arrive at the same one, so nothing in it is left to the compiler: the products
// and sums are not contracted but where `fmaf` says so, and conversions, quotients and `ceilf` are exact or round once.
// 48 paged sequences of 2047 .. 4096 tokens (32 heads of 128, rank 2): 67.7 us with equal counts (288 workgroups), 43.4 so.
// At head size 128 a range is a whole number of rounds of its four waves: one of a round and a bit takes two, and a few more partials
// to merge (steps, us, any length / whole rounds: 24 x 1024 tokens, 32 heads 23.9 / 23.0, four tokens of 6 x 2048, 16 heads 23.4 / 22.7, 4 x
// 8192, 32 heads 24.2 / 23.4, 48 x 4096 50.4 / 50.1).  At 64 a round is short and fewer workgroups weigh more (40 x 1024, 16 heads 18.6 / 18.9).
constexpr int kMaxPlanEntries = 64;
// What costs time in it is latency, twice per call (here and in the merge): sums over the lanes go through DPP adds (through
// the LDS permute they were 1 400 cycles), and the search takes four instructions per entry.  With both, append, decode and
// merge of the step above 57.1 -> 54.1 us, of 6 sequences of 1022 .. 2048 tokens with four query tokens each 26.1 -> 24.8.
template <int CTRL, int ROWS>
__device__ __forceinline__ int add_from(int x) { return x + __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false); }
__device__ __forceinline__ int wave_prefix_sum(int x) {  // lane i: sum of lanes 0 .. i
  x = add_from<0x111, 0xf>(x);  // row_shr 1, 2, 4, 8: inside rows of 16 lanes
  x = add_from<0x112, 0xf>(x);
  x = add_from<0x114, 0xf>(x);
  x = add_from<0x118, 0xf>(x);
  x = add_from<0x142, 0xa>(x);  // row_bcast 15: the last lane of rows 0 and 2 to rows 1 and 3
  return add_from<0x143, 0xc>(x);  // row_bcast 31: lane 31 to rows 2 and 3
}
struct RangePlan { int S, first; };  // of batch entry `lane`: its number of ranges and the first one's index
__device__ __forceinline__ RangePlan plan_ranges(const int32_t* kvlen, int B, int lk, int slots, float round_keys, float min_keys) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int len = lane < B ? max(0, min(kvlen[lane], lk)) : 0;
  const int total = __builtin_amdgcn_readlane(wave_prefix_sum(len), 63);
  const float shortest = fmaxf((float)total / (float)slots, min_keys);
  const float longest = slots > B ? fmaxf((float)total / (float)(slots - B) + 1.f, shortest) : (float)lk;
  float length = fmaf((longest - shortest) * (float)lane, 1.f / 63.f, shortest);
  if (round_keys > 0.f) length = ceilf(length / round_keys) * round_keys;
  const float inv = 1.f / length;
  // eight entries at a time, their chains side by side; an entry without keys counts as one of one key (one range), and so do
  // the lanes past the last entry, which are taken off again
  const uint32_t keys = __float_as_uint((float)max(len, 1));
  float count[8] = {};
  int j0 = 0;
  for (; j0 < B; j0 += 8)
#pragma unroll
    for (int j = 0; j < 8; ++j) count[j] += ceilf(__uint_as_float(__builtin_amdgcn_readlane(keys, j0 + j)) * inv);
  const int total_count = (int)(((count[0] + count[1]) + (count[2] + count[3])) + ((count[4] + count[5]) + (count[6] + count[7]))) - (j0 - B);
  const uint64_t fits = __ballot(total_count <= slots);
  RangePlan r;
  r.S = lane < B ? 1 : 0;
  if (fits) {
    const float pick = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(inv), __builtin_ctzll(fits)));
    if (lane < B) r.S = max(1, (int)ceilf((float)len * pick));
  }
  r.first = wave_prefix_sum(r.S) - r.S;
  return r;
}

// Range index -> batch entry, its range and its number of ranges; false past the last range.
__device__ __forceinline__ bool range_of(const DecodeParams& p, int x, int& b, int& split, int& S) {
  if (p.slots == 0) {
    S = p.S;
    b = x / S;
    split = x - b * S;
    return x < p.B * S;
  }
  const RangePlan plan = plan_ranges(p.kvlen, p.B, p.lk, p.slots, p.round_keys, p.min_keys);
  const int lane = threadIdx.x & 63;
  b = __popcll(__ballot(lane < p.B && plan.first <= x)) - 1;
  S = __builtin_amdgcn_readlane(plan.S, b);
  split = x - __builtin_amdgcn_readlane(plan.first, b);
  return split < S;
}

// Qm^T fragments (B operand of S'^T = B_k Qm^T): lane (h, g) holds Qm[h][16 ks + 8 g + 0..7] with
// Qm[h, :] = scale * sum_r qa[r, h] qb[r, :], itself a product of the matrix cores (rows d, columns h, contraction over
// the ranks in steps of 16, zeros past the last).  `QRaw` holds the operands of one step as loaded, so that the loads can
// be issued ahead of the cache's.  An accumulator column has d = 8 q + 4 g + e of its block; exchanging halves between
// the packed words of neighbouring q gives the order of the fragments.
// (On the vector ALU this took 8 600 of the 35 800 cycles of a decode of 1500 keys, half of them the conversions; with this
// form and the merge of the waves in 16-byte words, 64 x 8192 keys: 112.1 -> 107.3 us.)
// Both operands have the ranks innermost, which memory has not: the token factors come as whole rows, 16 bytes a lane, and are
// transposed by the reads of the wave's LDS region (laid out as the cache's rows are, in `lds`), the head factors two bytes at a
// time: 6 loads a lane for a rank of 6 where two bytes at a time for both took 40.  Slot (g, j) of a fragment is rank 8 (j / 4) + 4 g + j % 4 of the step, in both; steps of up to 8 ranks load half of it.
template <int D>
struct QRaw { uint16_t a[8]; u32x4 b[D / 32]; };
template <int D>
__device__ __forceinline__ QRaw<D> load_q_factors(const uint16_t* ap, int64_t a_stride, const uint16_t* bp, int64_t b_stride, int r0, int rq, int l) {
  constexpr int CPR = D / 8, RPI = 64 / CPR;
  const int g = l >> 5;
  QRaw<D> raw = {};
  // reads past the last rank repeat it and count as zero
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (half && r0 + 8 >= rq) break;
#pragma unroll
    for (int n = half * D / 64; n < (half + 1) * D / 64; ++n)
      raw.b[n] = *reinterpret_cast<const u32x4*>(bp + min(r0 + n * RPI + l / CPR, rq - 1) * b_stride + 8 * (l % CPR));
    const uint16_t* pa = ap + min(r0 + 8 * half + 4 * g, rq - 1) * a_stride;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      raw.a[4 * half + j] = *pa;
      pa += r0 + 8 * half + 4 * g + j + 1 < rq ? a_stride : 0;
    }
  }
  return raw;
}

// Where a lane's pieces of a tile of rows of D lie in LDS (elements; 16-byte chunk c of row r at chunk c ^ (r mod chunks)): one
// address each, from which the others differ by an exclusive or with a constant, a constant, or both.
template <int D>
struct TileAt {
  static constexpr int CPR = D / 8, RPI = 64 / CPR;
  int wr, row, tr;
  __device__ __forceinline__ explicit TileAt(int l) {
    const int i = l & 31, g = l >> 5, lp = l & 15, dhalf = (l >> 4) & 1, r = 4 * g + (lp >> 2);
    wr = (l / CPR) * D + 8 * ((l % CPR) ^ (l / CPR));
    row = i * D + 8 * (g ^ (i & (CPR - 1)));
    tr = r * D + 8 * ((2 * dhalf + ((lp & 3) >> 1)) ^ r) + 4 * (lp & 1);
  }
  __device__ __forceinline__ int write(int n) const { return (wr ^ (8 * ((n * RPI) & (CPR - 1)))) + n * RPI * D; }  // row n RPI + l / CPR, chunk l % CPR
  __device__ __forceinline__ int read(int ks) const { return row ^ (16 * ks); }                                    // row i, chunk 2 ks + g
  // transposed: rows 16 kk + 8 hi + 4 g + 0..3, columns 32 db + 0..31
  __device__ __forceinline__ int read_tr(int kk, int hi, int db) const { return (tr ^ (32 * db) ^ (hi && CPR == 16 ? 64 : 0)) + (16 * kk + 8 * hi) * D; }
};
template <int D>
__device__ __forceinline__ bf16x8 tile_tr(const uint16_t* tile, const TileAt<D>& at, int kk, int db) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(tile + at.read_tr(kk, 0, db)));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(tile + at.read_tr(kk, 1, db)));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int D>
__device__ __forceinline__ void finish_q_fragments(QRaw<D> raw, const uint16_t* ap, int64_t a_stride, const uint16_t* bp, int64_t b_stride,
                                                   int rq, float scale, int l, uint16_t* lds, const TileAt<D>& at, bf16x8 (&qf)[D / 16]) {
  constexpr int NDB = D / 32, NKS = D / 16, CPR = D / 8, RPI = 64 / CPR;
  const int g = l >> 5;
  f32x16 acc[NDB];
  auto step = [&](int r0, auto first_c) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < D / 32; ++n)
      *reinterpret_cast<u32x4*>(lds + at.write(n)) = r0 + n * RPI + l / CPR < rq ? raw.b[n] : u32x4{0, 0, 0, 0};
    u32x4 aw;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = r0 + 8 * (j >> 1) + 4 * g + 2 * (j & 1);
      aw[j] = (r < rq ? (uint32_t)raw.a[2 * j] : 0u) | (r + 1 < rq ? (uint32_t)raw.a[2 * j + 1] << 16 : 0u);
    }
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      f32x16 c;
#pragma unroll
      for (int v = 0; v < 16; ++v) c[v] = decltype(first_c)::value ? 0.f : acc[db][v];
      acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tile_tr<D>(lds, at, 0, db), __builtin_bit_cast(bf16x8, aw), c, 0, 0, 0);
    }
  };
  step(0, std::true_type{});
  for (int r0 = 16; r0 < rq; r0 += 16) {
    raw = load_q_factors<D>(ap, a_stride, bp, b_stride, r0, rq, l);
    step(r0, std::false_type{});
  }
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = pack_bf16(acc[ks / 2][8 * (ks & 1) + 2 * j] * scale, acc[ks / 2][8 * (ks & 1) + 2 * j + 1] * scale);
    const auto even = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
    const auto odd = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
    qf[ks] = __builtin_bit_cast(bf16x8, u32x4{even[0], odd[0], even[1], odd[1]});
  }
}

template <int D>
struct DecodeLds {
  static constexpr int kB = kRowsPerBlock * D;       // elements of one B tile
  static constexpr int kA = kRowsPerBlock * 32;      // elements of one A tile (32 heads)
  static constexpr int kWave = 2 * kB + 2 * kA;      // elements per wave
  static constexpr int kRedStride = D + 4;           // fp32 row stride of the wave-merge staging (spreads the banks)
  static constexpr int kReduce = 32 * kRedStride * 2 + 128;  // fp32 O^T + m + l, in uint16 units
  static constexpr int kPerWave = kWave > kReduce ? kWave : kReduce;
  static constexpr size_t kBytes = (size_t)kWaves * kPerWave * sizeof(uint16_t);
  // with several query rows per workgroup: plus their Q fragments (NQ sets x D/16 steps x 64 lanes x 16 bytes)
  static constexpr size_t bytes(int nq, bool side) { return kBytes + (nq > 1 || side ? (size_t)nq * (D / 16) * 64 * 16 : 0); }
};

// At head size 64 and from rank 4 on two workgroups fit a compute unit, which the compiler has to be told: at 258 registers
// instead of 256 rank 8 lost the second one (64 heads, two rows per workgroup: 48 x 4096 keys, eight rows 544 -> 707 us; 4 x 1024
// rows and keys without K and V 2.42 -> 3.15 ms; 2.10 so, with 204).
// So it is with rows side by side at every rank: 256 to 260 registers at ranks 1 and 2, three of four instances without the second
// workgroup (us, 16 heads, before / now: 300 x 1000 keys, rank 1, two rows 34.0 / 28.5; 64 x 8192, rank 2, four rows 75.0 / 68.7; 4 x 8192 13.4 / 12.6).
constexpr int min_waves(int d, int rk, bool side) { return d == 64 && (rk >= 4 || side) ? 2 : 1; }
template <int D, int RK, bool PAGED, int NQ, Reads READS, bool SIDE = false>
__global__ __launch_bounds__(kWaves * 64, min_waves(D, RK, SIDE)) void decode_kernel(DecodeParams p) {
  constexpr int CPR = D / 8;               // 16-byte chunks per B row
  constexpr int RPI = 64 / CPR;            // B rows per load instruction
  constexpr int NLB = kRowsPerBlock / RPI; // load instructions per B tile
  constexpr int NKS = D / 16;
  constexpr int NDB = D / 32;
  constexpr int NTOK = RK <= 4 ? 16 / RK : 32 / RK;  // tokens whose rows this lane holds, per block
  constexpr int NV = RK <= 4 ? RK : RK / 2;          // rows of one token held by this half of the wave
  static_assert(RK == 1 || RK == 2 || RK == 4 || RK == 8 || RK == 16 || RK == 32, "a block of 32 rows holds whole tokens");

  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];

  // workgroup id -> (key range x, query row qi): ids are dealt to the 8 XCDs round-robin, and the
  // rows of one query token group read the same cache slice, so they get ids that are 8 apart
  // (same XCD, same L2) and next to each other in launch order (resident together)
  // A workgroup serves NQ column sets from one pass over its cache blocks (each staged block is used NQ times).  A set is
  // the heads of one query row, or (SIDE: 8 or 16 heads) those of 32 / H rows side by side in the 32 columns; rows past the
  // last one repeat it and are not stored.
  const int rps = SIDE ? 32 / p.H : 1;            // rows per set
  const int rpw = NQ * rps;                       // rows per workgroup
  const int nqg = (p.lq + rpw - 1) / rpw;         // groups of as many query rows
  const int gid = blockIdx.x, grp = gid / (8 * nqg), rem = gid - grp * 8 * nqg;
  const int qi0 = rpw * (rem >> 3), x = grp * 8 + (rem & 7);
  int b, split, S;
  if (!range_of(p, x, b, split, S)) return;  // the grid is rounded up to whole groups of 8 ranges
  const int h0 = blockIdx.y * 32;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
  const int ci = SIDE ? i / p.H : 0;                           // this lane's row of a set
  const int hl = SIDE ? i - ci * p.H : min(h0 + i, p.H - 1);  // and its head (clamped: lanes past H idle along)

  uint16_t* lds = smem + w * DecodeLds<D>::kPerWave;
  uint16_t* lds_bk = lds;
  uint16_t* lds_bv = lds + DecodeLds<D>::kB;
  uint16_t* lds_ak = lds + 2 * DecodeLds<D>::kB;
  uint16_t* lds_av = lds_ak + DecodeLds<D>::kA;

  const TileAt<D> at(l);

  // ---- Qm^T fragments: requested ahead of the cache's first blocks, finished while those are in flight.
  // With one query row they stay in registers; with several (no more than waves) wave r builds row r's fragments once
  // and parks them in LDS behind the waves' staging regions (fragment (set, ks) of lane l at
  // [(set NKS + ks) 64 + l], written by the lanes whose row it is: another row's infinities never
  // meet theirs), from where every wave reads them: one set into its registers, two as it needs them,
  // when the registers go to the accumulators instead.
  static_assert(!SIDE || NQ == 1, "rows side by side are one set");
  bf16x8 qf[NQ == 1 ? NKS : 1];
  u32x4* const lds_q = reinterpret_cast<u32x4*>(smem + kWaves * DecodeLds<D>::kPerWave);
  const int qi_build = NQ == 1 && !SIDE ? qi0 : min(qi0 + w, p.lq - 1);
  const uint16_t* const qa_row = static_cast<const uint16_t*>(p.qa.ptr) + b * p.qa.stride_b + (int64_t)qi_build * p.qa.stride_l + hl;
  const uint16_t* const qb_row = static_cast<const uint16_t*>(p.qb.ptr) + b * p.qb.stride_b + (int64_t)qi_build * p.qb.stride_l;
  auto build_q = [&](const QRaw<D>& raw) __attribute__((always_inline)) {
    if constexpr (NQ == 1 && !SIDE) {
      finish_q_fragments<D>(raw, qa_row, p.qa.stride_r, qb_row, p.qb.stride_r, p.rq, p.qscale, l, lds, at, qf);
    } else {
      if (w < rpw) {
        bf16x8 tmp[NKS];
        finish_q_fragments<D>(raw, qa_row, p.qa.stride_r, qb_row, p.qb.stride_r, p.rq, p.qscale, l, lds, at, tmp);
        if (!SIDE || ci == w) {
#pragma unroll
          for (int ks = 0; ks < NKS; ++ks) lds_q[((SIDE ? 0 : w) * NKS + ks) * 64 + l] = __builtin_bit_cast(u32x4, tmp[ks]);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the cache's loads stay in flight
      if constexpr (NQ == 1) {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) qf[ks] = __builtin_bit_cast(bf16x8, lds_q[ks * 64 + l]);
      }
    }
  };

  // ---- this wave's blocks: part, part + nparts, part + 2 nparts, ... (dealt round robin, so the
  // waves of the grid, which advance in step, read neighbouring addresses at any one time)
  const int nparts = S * kWaves;
  const int part = split * kWaves + w;
  // keys of this batch entry that each query row sees, and the most any of them sees
  const int len_all = p.kvlen ? min(p.kvlen[b], p.lk) : p.lk;
  int row_last[NQ], len_b = 0;
#pragma unroll
  for (int r = 0; r < NQ; ++r) {
    auto keys_of = [&](int row) { return max(0, min(len_all, min(row, p.lq - 1) + p.climit + (p.cbr ? len_all - p.lq_total : 0))); };
    row_last[r] = keys_of(qi0 + r * rps + ci) * RK - 1;
    len_b = max(len_b, keys_of(qi0 + r * rps + rps - 1));  // a row sees no fewer keys than the one before it
  }
  const int blk_begin = part;
  const int blk_end = (len_b * RK + kRowsPerBlock - 1) / kRowsPerBlock;  // 32-row blocks of its cache
  const int blk_step = nparts;
  const int last_row = len_b * RK - 1;

  // rows of the cache matrices: row = token * RK + rank, row stride = stride_r
  // (paged cache: the arrays are page pools, stride_b = elements between pages, and a block of 32
  // rows lies inside one page, which the page table of this batch entry locates)
  const int64_t boff = PAGED ? 0 : b;
  const uint16_t* kb_base = static_cast<const uint16_t*>(p.kb.ptr) + boff * p.kb.stride_b;
  const uint16_t* vb_base = static_cast<const uint16_t*>(p.vb.ptr) + boff * p.vb.stride_b;
  const uint16_t* ka_base = static_cast<const uint16_t*>(p.ka.ptr) + boff * p.ka.stride_b + h0;
  const uint16_t* va_base = static_cast<const uint16_t*>(p.va.ptr) + boff * p.va.stride_b + h0;
  const int rpp = PAGED ? p.page_size * RK : 1;  // rows per page
  const int a_chunks = min(4, (p.H - h0) / 8);  // valid 16-byte chunks of an A row in this head block

  // loader lane roles
  const int lb_row = l / CPR, lb_c = l % CPR;             // B tiles: row within the instruction, chunk
  // A tiles: 16 rows per instruction; 8 or 16 heads with their rows side by side fill the 32 columns by repeating
  const int la_row = l >> 2, la_c = SIDE ? (l & 3) & (a_chunks - 1) : min(l & 3, a_chunks - 1);

  // two register sets: while one block is staged and consumed, two more are in flight (one set
  // with NQ rows, whose accumulators take the room and whose blocks take NQ times as long to
  // consume)
  constexpr int NSETS = NQ == 1 ? 2 : 1;
  u32x4 rbk[NSETS][NLB], rbv[NSETS][NLB], rak[NSETS][2], rav[NSETS][2];
  // Paged cache: the place of a block (its page, the row in it) is looked up one visit of its register set ahead (when the
  // set's previous block is requested), so that no request waits for a page-table entry
  struct Place { int32_t page; int row; };  // the page as loaded: made a scalar only where it is used, which waits for it
  Place ahead[NSETS] = {};
  auto lookup = [&](int blk) __attribute__((always_inline)) -> Place {
    if constexpr (!PAGED) return Place{0, 0};
    const int row0 = max(min(blk, blk_end - 1), 0) * kRowsPerBlock, page = p.page_shift >= 0 ? row0 >> p.page_shift : row0 / rpp;
    return Place{p.page_table[(int64_t)b * p.pages_per_seq + page], row0 - page * rpp};
  };
  // A block's rows are read through buffer resources that end with its last valid row (what lies past it reads as zero): the
  // lane's offset in a block never changes and the rest of an address is scalar.
  // Every request is made whether or not its block is there (a block past the last one has no rows: its resource is empty), and
  // there is no branch around a load: each path through the loop then has the same number of loads in flight, and the wait in
  // front of `stage` counts past the other set's.  Behind a branch they are waited for by the count of the path without them: to
  // the last one, and the second set is in flight in name only.
  // us per call, addresses per lane and load behind branches / this, 32 heads of 128, rank 2: 90 sequences of 6000 keys, two
  // rows, 136 / 125; 300 of 1000, one row, 100 / 95; 16 heads of 64: 20 of 12 345 31.8 / 30.7.  64 x 8192 keys (108 us) is bound
  // by HBM and has them alike; 40 paged sequences of 4800 - 9600 keys, 64 heads of 64, lose 2 % (77.7 / 79.4).
  const int kb_sr = 2 * (int)p.kb.stride_r, vb_sr = 2 * (int)p.vb.stride_r, ka_sr = 2 * (int)p.ka.stride_r, va_sr = 2 * (int)p.va.stride_r;
  const int kb_voff = lb_row * kb_sr + 16 * lb_c, vb_voff = lb_row * vb_sr + 16 * lb_c;
  const int ka_voff = la_row * ka_sr + 16 * la_c, va_voff = la_row * va_sr + 16 * la_c;
  auto issue = [&](auto set_c, int blk) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    const int row0 = blk * kRowsPerBlock;
    const int rows = max(0, min(kRowsPerBlock, last_row + 1 - row0));
    int64_t page = 0, first = row0;  // of a page pool: the page and the row in it
    if constexpr (PAGED) {
      page = last_row < 0 ? 0 : scalar(ahead[set].page);
      first = ahead[set].row;
      ahead[set] = lookup(blk + NSETS * blk_step);
    }
    const uint16_t* const kb = kb_base + page * p.kb.stride_b + first * p.kb.stride_r;
    const uint16_t* const vb = vb_base + page * p.vb.stride_b + first * p.vb.stride_r;
    const uint16_t* const ka = ka_base + page * p.ka.stride_b + first * p.ka.stride_r;
    const uint16_t* const va = va_base + page * p.va.stride_b + first * p.va.stride_r;
    if constexpr (READS == Reads::kFar) {
      auto row_at = [&](const uint16_t* base, int row, int64_t stride, int c) __attribute__((always_inline)) {
        return row < rows ? *reinterpret_cast<const u32x4*>(base + row * stride + 8 * c) : u32x4{0, 0, 0, 0};
      };
#pragma unroll
      for (int n = 0; n < NLB; ++n) {
        rbk[set][n] = row_at(kb, n * RPI + lb_row, p.kb.stride_r, lb_c);
        rbv[set][n] = row_at(vb, n * RPI + lb_row, p.vb.stride_r, lb_c);
      }
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        rak[set][n] = row_at(ka, 16 * n + la_row, p.ka.stride_r, la_c);
        rav[set][n] = row_at(va, 16 * n + la_row, p.va.stride_r, la_c);
      }
      return;
    }
    auto rows_of = [&](const uint16_t* base, int sr, int width) __attribute__((always_inline)) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), 0, rows > 0 ? (rows - 1) * sr + 2 * width : 0, kRsrcFlags);
    };
    const __amdgpu_buffer_rsrc_t kb_rs = rows_of(kb, kb_sr, D), vb_rs = rows_of(vb, vb_sr, D);
    const __amdgpu_buffer_rsrc_t ka_rs = rows_of(ka, ka_sr, 8 * a_chunks), va_rs = rows_of(va, va_sr, 8 * a_chunks);
    constexpr int aux = READS == Reads::kStreaming ? 2 : 0;  // bit 1: non-temporal
#pragma unroll
    for (int n = 0; n < NLB; ++n) {
      rbk[set][n] = __builtin_amdgcn_raw_buffer_load_b128(kb_rs, kb_voff, n * RPI * kb_sr, aux);
      rbv[set][n] = __builtin_amdgcn_raw_buffer_load_b128(vb_rs, vb_voff, n * RPI * vb_sr, aux);
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      rak[set][n] = __builtin_amdgcn_raw_buffer_load_b128(ka_rs, ka_voff, 16 * n * ka_sr, aux);
      rav[set][n] = __builtin_amdgcn_raw_buffer_load_b128(va_rs, va_voff, 16 * n * va_sr, aux);
    }
  };
  auto stage = [&](auto set_c) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int n = 0; n < NLB; ++n) {
      *reinterpret_cast<u32x4*>(lds_bk + at.write(n)) = rbk[set][n];
      *reinterpret_cast<u32x4*>(lds_bv + at.write(n)) = rbv[set][n];
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int row = 16 * n + la_row;
      *reinterpret_cast<u32x4*>(lds_ak + row * 32 + 8 * (l & 3)) = rak[set][n];
      *reinterpret_cast<u32x4*>(lds_av + row * 32 + 8 * (l & 3)) = rav[set][n];
    }
  };

  f32x16 o[NQ][NDB];
  float m[NQ], lsum[NQ];
#pragma unroll
  for (int r = 0; r < NQ; ++r) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[r][db][v] = 0.f;
    m[r] = -INFINITY;
    lsum[r] = 0.f;
  }

  const int lp = l & 15, dhalf = (l >> 4) & 1;

  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  ahead[0] = lookup(blk_begin);
  if constexpr (NSETS == 2) ahead[1] = lookup(blk_begin + blk_step);
  const QRaw<D> q_raw = load_q_factors<D>(qa_row, p.qa.stride_r, qb_row, p.qb.stride_r, 0, p.rq, l);
  __builtin_amdgcn_sched_barrier(0);  // in the order of their use, as in the loop: what is waited for is counted from the last one
  issue(Set0{}, blk_begin);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NSETS == 2) issue(Set1{}, blk_begin + blk_step);
  __builtin_amdgcn_sched_barrier(0);
  build_q(q_raw);

  auto compute = [&](int blk) {
    // ---- a_k / a_v of this lane's head for its 16 rows (rows 8q + 4g + 0..3, q = 0..3)
    float ak[16], av[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int arow = 8 * q + 4 * g + (lp >> 2);
      const s16x4 tk = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (s16x4 __attribute__((address_space(3)))*)(lds_ak + arow * 32 + 16 * dhalf + 4 * (lp & 3)));
      const s16x4 tv = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (s16x4 __attribute__((address_space(3)))*)(lds_av + arow * 32 + 16 * dhalf + 4 * (lp & 3)));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ak[4 * q + j] = bf16bits_to_f32((uint16_t)tk[j]);
        av[4 * q + j] = bf16bits_to_f32((uint16_t)tv[j]);
      }
    }
    const int row0 = blk * kRowsPerBlock;

#pragma unroll
    for (int r = 0; r < NQ; ++r) {
      // keep the rows' instruction streams apart: interleaved, their temporaries do not fit the registers
      if constexpr (NQ > 1) __builtin_amdgcn_sched_barrier(0);
      // ---- S'^T[row, h] = sum_d B_k[row, d] Qm[h, d]
      f32x16 sp;
#pragma unroll
      for (int v = 0; v < 16; ++v) sp[v] = 0.f;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(lds_bk + at.read(ks));
        if constexpr (NQ == 1) {
          sp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], sp, 0, 0, 0);
        } else {
          const bf16x8 qv = __builtin_bit_cast(bf16x8, lds_q[(r * NKS + ks) * 64 + l]);
          sp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qv, sp, 0, 0, 0);
        }
      }

      // ---- logits per token (log2 domain), masked past the keys this query row sees
      // (a token's RK rows are registers v0 .. v0 + NV - 1; from rank 8 on they span both halves of
      // the wave, which then hold the same tokens and exchange their partial sums)
      float st[NTOK];
      float tmax = -INFINITY;
#pragma unroll
      for (int t = 0; t < NTOK; ++t) {
        const int v0 = t * NV;
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j) acc += ak[v0 + j] * sp[v0 + j];
        if constexpr (RK >= 8) acc = halves_sum(acc);
        const int row = RK >= 8 ? row0 + RK * t : row0 + 8 * (v0 >> 2) + 4 * g + (v0 & 3);  // the token's first row
        if (row > row_last[r]) acc = -INFINITY;
        st[t] = acc;
        tmax = fmaxf(tmax, acc);
      }
      tmax = halves_max(tmax);
      // finite with one query row (row0 itself is always inside its keys); a row that sees fewer
      // keys than its neighbour can meet a block with none of its keys, before any or after all.
      // The reference is a whole number (the running maximum rounded up): 2^(s - m) then has the same
      // significand whatever m is, so the bf16 rounding of P' below does not depend on how the keys are
      // split over waves and ranges, and every rescaling factor (here, in the wave merge, in the merge of
      // the key ranges) is an exact power of two
      const float m_new = fmaxf(m[r], __builtin_ceilf(tmax));
      const float m_use = (NQ > 1 || SIDE) && m_new == -INFINITY ? 0.f : m_new;
      if (NQ == 1 && blk == blk_begin) {
        m[r] = m_new;  // nothing to rescale yet
      } else if (__any(m_new > m[r])) {
        const float alpha = __builtin_amdgcn_exp2f(m[r] - m_use);
        lsum[r] *= alpha;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int v = 0; v < 16; ++v) o[r][db][v] *= alpha;
        m[r] = m_new;
      }

      // ---- P'^T[row, h] = p[h, token(row)] * a_v[row, h], packed as the B operand of the PV product
      float pp[16];
#pragma unroll
      for (int t = 0; t < NTOK; ++t) {
        const float pt = __builtin_amdgcn_exp2f(st[t] - m_use);
        lsum[r] += RK >= 8 ? 0.5f * pt : pt;  // both halves hold the token: each adds half of it
#pragma unroll
        for (int j = 0; j < NV; ++j) pp[t * NV + j] = pt * av[t * NV + j];
      }
      bf16x8 pf[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        u32x4 pk;
#pragma unroll
        for (int j = 0; j < 4; ++j) pk[j] = pack_bf16(pp[8 * kk + 2 * j], pp[8 * kk + 2 * j + 1]);
        pf[kk] = __builtin_bit_cast(bf16x8, pk);
      }

      // ---- O^T[d, h] += sum_row B_v[row, d] P'^T[row, h]; slot (g, j) = row 16kk + 8(j/4) + 4g + j%4
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
          o[r][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tile_tr<D>(lds_bv, at, kk, db), pf[kk], o[r][db], 0, 0, 0);
      }
    }
  };

  if constexpr (NSETS == 2) {
    int blk = blk_begin;
    for (; blk + blk_step < blk_end; blk += 2 * blk_step) {  // left in one place, for the same reason
      stage(Set0{});
      issue(Set0{}, blk + 2 * blk_step);
      compute(blk);
      stage(Set1{});
      issue(Set1{}, blk + 3 * blk_step);
      compute(blk + blk_step);
    }
    if (blk < blk_end) {
      stage(Set0{});
      compute(blk);
    }
  } else {
    for (int blk = blk_begin; blk < blk_end; blk += blk_step) {
      stage(Set0{});
      issue(Set0{}, blk + blk_step);
      compute(blk);
    }
  }

  // ---- merge the 4 waves through LDS (each wave reuses its own staging region), row by row
  constexpr int RS = DecodeLds<D>::kRedStride;
  float* red_o = reinterpret_cast<float*>(lds);  // [32 heads][RS]
  float* red_m = red_o + 32 * RS;
  float* red_l = red_m + 32;
#pragma unroll
  for (int r = 0; r < NQ; ++r) {
    const int qr = qi0 + r * rps;
    if (qr >= p.lq) break;  // uniform: a set of repeated rows
    const int nh = SIDE ? min(32, (p.lq - qr) * p.H) : min(32, p.H - h0);  // columns that are stored: heads, or (row, head)
    const float ltot = halves_sum(lsum[r]);
    __syncthreads();  // the staging (or the previous row's merge) has been read by every wave
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq)
        *reinterpret_cast<f32x4*>(red_o + i * RS + 32 * db + 8 * vq + 4 * g) =
            f32x4{o[r][db][4 * vq], o[r][db][4 * vq + 1], o[r][db][4 * vq + 2], o[r][db][4 * vq + 3]};
    if (g == 0) {
      red_m[i] = m[r];
      red_l[i] = ltot;
    }
    __syncthreads();

    const int64_t pbase = ((int64_t)x * p.lq + qr) * p.H + h0;
#pragma unroll(NQ == 1 ? 4 : 1)
    for (int idx = tid; idx < nh * (D / 4); idx += kWaves * 64) {
      const int hh = idx / (D / 4), d = 4 * (idx % (D / 4));
      float mw[kWaves], mmax = -INFINITY;
#pragma unroll
      for (int ww = 0; ww < kWaves; ++ww) {
        mw[ww] = reinterpret_cast<const float*>(smem + ww * DecodeLds<D>::kPerWave)[32 * RS + hh];
        mmax = fmaxf(mmax, mw[ww]);
      }
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      float lacc = 0.f;
#pragma unroll
      for (int ww = 0; ww < kWaves; ++ww) {
        const float* ro = reinterpret_cast<const float*>(smem + ww * DecodeLds<D>::kPerWave);
        const float f = mw[ww] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[ww] - mmax);
        acc += f * *reinterpret_cast<const f32x4*>(ro + hh * RS + d);
        lacc += f * ro[32 * RS + 32 + hh];
      }
      *reinterpret_cast<f32x4*>(p.part_o + (pbase + hh) * D + d) = acc;
      if (d == 0) {
        p.part_m[pbase + hh] = mmax;
        p.part_l[pbase + hh] = lacc;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The same decode for an fp32 cache (the reference's default dtype): fp32 MFMA contractions
// (v_mfma_f32_32x32x2_f32) on fp32 rows.  Same decomposition and the same workspace; what differs
// is the operand order a two-index fp32 step asks for: over d, wave half g takes d = 8m + 4g + e
// (one 16-byte LDS read feeds four steps); over the block's rows, half g takes the row its S'^T
// register belongs to, and the 32 rows of block db of O^T are d = (D/32) i + db, so one 16-byte
// read of B_v[row][(D/32) i ...] feeds every block.  One block of loads is in flight in registers
// (128 of them for D = 128) while the previous block is consumed; the head factors a_k, a_v are
// read straight into the registers of the logits they multiply.
template <int D>
struct DecodeF32Lds {
  static constexpr int RS = D + 4;                   // row stride (floats)
  static constexpr int kTile = kRowsPerBlock * RS;   // one B tile
  static constexpr int kPerWave = 2 * kTile;         // B_k and B_v; the wave merge reuses it (32 x RS + 64 floats)
  static constexpr size_t kBytes = (size_t)kWaves * kPerWave * sizeof(float);
};

template <int D, int RK, bool PAGED>
__global__ __launch_bounds__(kWaves * 64) void decode_f32_kernel(DecodeParams p) {
  constexpr int CPR = D / 4;               // 16-byte chunks per B row
  constexpr int RPI = 64 / CPR;            // B rows per load instruction
  constexpr int NLB = kRowsPerBlock / RPI; // load instructions per B tile
  constexpr int NDB = D / 32;
  constexpr int NTOK = RK <= 4 ? 16 / RK : 32 / RK;  // tokens whose rows this lane holds, per block
  constexpr int NV = RK <= 4 ? RK : RK / 2;          // rows of one token held by this half of the wave
  constexpr int RS = DecodeF32Lds<D>::RS;
  static_assert(RK == 1 || RK == 2 || RK == 4 || RK == 8 || RK == 16 || RK == 32, "a block of 32 rows holds whole tokens");
  typedef __attribute__((ext_vector_type(NDB))) float f32xN;

  extern __shared__ __attribute__((aligned(16))) float smem_dec_f32[];

  // workgroup id -> (key range x, query row qi): ids are dealt to the 8 XCDs round-robin, and the
  // rows of one query token group read the same cache slice, so they get ids that are 8 apart
  // (same XCD, same L2) and next to each other in launch order (resident together)
  const int gid = blockIdx.x, grp = gid / (8 * p.lq), rem = gid - grp * 8 * p.lq;
  const int qi = rem >> 3, x = grp * 8 + (rem & 7);
  int b, split, S;
  if (!range_of(p, x, b, split, S)) return;  // the grid is rounded up to whole groups of 8 ranges
  const int h0 = blockIdx.y * 32;
  const int tid = threadIdx.x;
  const int w = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int hl = min(h0 + i, p.H - 1);  // this lane's head (clamped: lanes past H idle along)

  float* const lds = smem_dec_f32 + w * DecodeF32Lds<D>::kPerWave;
  float* const lds_bk = lds;
  float* const lds_bv = lds + DecodeF32Lds<D>::kTile;

  const int nparts = S * kWaves;
  const int part = split * kWaves + w;
  const int len_all = p.kvlen ? min(p.kvlen[b], p.lk) : p.lk;
  const int len_b = max(0, min(len_all, qi + p.climit + (p.cbr ? len_all - p.lq_total : 0)));
  const int blk_begin = part;
  const int blk_end = (len_b * RK + kRowsPerBlock - 1) / kRowsPerBlock;
  const int blk_step = nparts;
  const int last_row = len_b * RK - 1;

  // (paged cache: the arrays are page pools, stride_b = elements between pages, and a block of 32
  // rows lies inside one page, which the page table of this batch entry locates)
  const int64_t boff = PAGED ? 0 : b;
  const float* const kb_base = static_cast<const float*>(p.kb.ptr) + boff * p.kb.stride_b;
  const float* const vb_base = static_cast<const float*>(p.vb.ptr) + boff * p.vb.stride_b;
  const float* const ka_base = static_cast<const float*>(p.ka.ptr) + boff * p.ka.stride_b + hl;
  const float* const va_base = static_cast<const float*>(p.va.ptr) + boff * p.va.stride_b + hl;
  const int rpp = PAGED ? p.page_size * RK : 1;  // rows per page
  const int lb_row = l / CPR, lb_c = l % CPR;

  // one register set: the block after the one being consumed
  f32x4 rbk[NLB], rbv[NLB];
  float rak[16], rav[16];
  // (paged cache: a block's page is looked up while the block before it is requested)
  auto lookup = [&](int blk) __attribute__((always_inline)) -> int32_t {
    return PAGED && blk < blk_end ? p.page_table[(int64_t)b * p.pages_per_seq + blk * kRowsPerBlock / rpp] : 0;
  };
  int32_t page_ahead = lookup(blk_begin);
  auto issue = [&](int blk) {
    const int row0 = blk * kRowsPerBlock;
    // element offsets that take a logical row of this block to its place in the page pool
    int64_t pkb = 0, pvb = 0, pka = 0, pva = 0;
    if constexpr (PAGED) {
      const int page = row0 / rpp;
      const int64_t phys = page_ahead;
      page_ahead = lookup(blk + blk_step);
      const int64_t first = (int64_t)page * rpp;  // first logical row of the page
      pkb = phys * p.kb.stride_b - first * p.kb.stride_r;
      pvb = phys * p.vb.stride_b - first * p.vb.stride_r;
      pka = phys * p.ka.stride_b - first * p.ka.stride_r;
      pva = phys * p.va.stride_b - first * p.va.stride_r;
    }
#pragma unroll
    for (int n = 0; n < NLB; ++n) {
      const int row = min(row0 + n * RPI + lb_row, last_row);
      rbk[n] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(kb_base + pkb + (int64_t)row * p.kb.stride_r + 4 * lb_c));
      rbv[n] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(vb_base + pvb + (int64_t)row * p.vb.stride_r + 4 * lb_c));
    }
    // a[row][head of this lane] for the 16 rows this lane's S'^T registers belong to
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = min(row0 + 8 * (v >> 2) + 4 * g + (v & 3), last_row);
      rak[v] = ka_base[pka + (int64_t)row * p.ka.stride_r];
      rav[v] = va_base[pva + (int64_t)row * p.va.stride_r];
    }
  };
  float ak[16], av[16];
  auto stage = [&]() {
#pragma unroll
    for (int n = 0; n < NLB; ++n) {
      const int row = n * RPI + lb_row;
      *reinterpret_cast<f32x4*>(lds_bk + row * RS + 4 * lb_c) = rbk[n];
      *reinterpret_cast<f32x4*>(lds_bv + row * RS + 4 * lb_c) = rbv[n];
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) { ak[v] = rak[v]; av[v] = rav[v]; }
  };

  if (blk_begin < blk_end) issue(blk_begin);

  // ---- Qm (B operand of S'^T = B_k Qm^T): qf[4m + e] = qscale * sum_r qa[r][h] qb[r][8m + 4g + e]
  float qf[D / 2];
#pragma unroll
  for (int j = 0; j < D / 2; ++j) qf[j] = 0.f;
  {
    const float* ap = static_cast<const float*>(p.qa.ptr) + b * p.qa.stride_b + (int64_t)qi * p.qa.stride_l + hl;
    const float* bp = static_cast<const float*>(p.qb.ptr) + b * p.qb.stride_b + (int64_t)qi * p.qb.stride_l + 4 * g;
    for (int r = 0; r < p.rq; ++r) {
      const float a = ap[r * p.qa.stride_r];
#pragma unroll
      for (int m = 0; m < D / 8; ++m) {
        const f32x4 bv = *reinterpret_cast<const f32x4*>(bp + r * p.qb.stride_r + 8 * m);
#pragma unroll
        for (int e = 0; e < 4; ++e) qf[4 * m + e] += a * bv[e];
      }
    }
#pragma unroll
    for (int j = 0; j < D / 2; ++j) qf[j] *= p.qscale;
  }

  f32x16 o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[db][v] = 0.f;
  float m = -INFINITY, lsum = 0.f;

  auto compute = [&](int blk) {
    // ---- S'^T[row, h] = sum_d B_k[row, d] Qm[h, d]; two accumulation chains, added at the end
    f32x16 sp, sp2;
#pragma unroll
    for (int v = 0; v < 16; ++v) { sp[v] = 0.f; sp2[v] = 0.f; }
#pragma unroll
    for (int mm = 0; mm < D / 8; ++mm) {
      const f32x4 kf = *reinterpret_cast<const f32x4*>(lds_bk + i * RS + 8 * mm + 4 * g);
      sp = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[0], qf[4 * mm], sp, 0, 0, 0);
      sp2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[1], qf[4 * mm + 1], sp2, 0, 0, 0);
      sp = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[2], qf[4 * mm + 2], sp, 0, 0, 0);
      sp2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[3], qf[4 * mm + 3], sp2, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) sp[v] += sp2[v];

    // ---- logits per token (log2 domain), masked past the end of the cache
    // (a token's RK rows are registers v0 .. v0 + NV - 1; from rank 8 on they span both halves of
    // the wave, which then hold the same tokens and exchange their partial sums)
    float st[NTOK];
    float tmax = -INFINITY;
    const int row0 = blk * kRowsPerBlock;
#pragma unroll
    for (int t = 0; t < NTOK; ++t) {
      const int v0 = t * NV;
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < NV; ++j) acc += ak[v0 + j] * sp[v0 + j];
      if constexpr (RK >= 8) acc = halves_sum(acc);
      const int row = RK >= 8 ? row0 + RK * t : row0 + 8 * (v0 >> 2) + 4 * g + (v0 & 3);  // the token's first row
      if (row > last_row) acc = -INFINITY;
      st[t] = acc;
      tmax = fmaxf(tmax, acc);
    }
    tmax = halves_max(tmax);
    const float m_new = fmaxf(m, tmax);  // finite: row0 itself is always inside the cache
    if (__any(m_new > m)) {
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      lsum *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[db][v] *= alpha;
      m = m_new;
    }

    // ---- P'^T[row, h] = p[h, token(row)] * a_v[row, h], in place of the logits' registers
    float pp[16];
#pragma unroll
    for (int t = 0; t < NTOK; ++t) {
      const float pt = __builtin_amdgcn_exp2f(st[t] - m);
      lsum += RK >= 8 ? 0.5f * pt : pt;  // both halves hold the token: each adds half of it
#pragma unroll
      for (int j = 0; j < NV; ++j) pp[t * NV + j] = pt * av[t * NV + j];
    }

    // ---- O^T[d, h] += sum_row B_v[row, d] P'^T[row, h]
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = 8 * (v >> 2) + 4 * g + (v & 3);
      const f32xN vf = *reinterpret_cast<const f32xN*>(lds_bv + row * RS + NDB * i);
#pragma unroll
      for (int db = 0; db < NDB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[db], pp[v], o[db], 0, 0, 0);
    }
  };

  for (int blk = blk_begin; blk < blk_end; blk += blk_step) {
    stage();  // waits for this block's loads; its registers are then free again
    if (blk + blk_step < blk_end) issue(blk + blk_step);
    compute(blk);
  }

  // ---- merge the 4 waves through LDS (each wave reuses its own staging region)
  const float ltot = halves_sum(lsum);
  float* red_o = lds;  // [32 heads][RS]: row 8 (v/4) + 4 g + v%4 of block db is d = NDB * row + db
  float* red_m = red_o + 32 * RS;
  float* red_l = red_m + 32;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = 8 * (v >> 2) + 4 * g + (v & 3);
    f32xN out;
#pragma unroll
    for (int db = 0; db < NDB; ++db) out[db] = o[db][v];
    *reinterpret_cast<f32xN*>(red_o + i * RS + NDB * row) = out;
  }
  if (g == 0) {
    red_m[i] = m;
    red_l[i] = ltot;
  }
  __syncthreads();

  const int nh = min(32, p.H - h0);
  const int64_t pbase = ((int64_t)x * p.lq + qi) * p.H + h0;
  for (int idx = tid; idx < nh * D; idx += kWaves * 64) {
    const int hh = idx / D, d = idx % D;
    float mw[kWaves], mmax = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < kWaves; ++ww) {
      mw[ww] = (smem_dec_f32 + ww * DecodeF32Lds<D>::kPerWave)[32 * RS + hh];
      mmax = fmaxf(mmax, mw[ww]);
    }
    float acc = 0.f, lacc = 0.f;
#pragma unroll
    for (int ww = 0; ww < kWaves; ++ww) {
      const float* ro = smem_dec_f32 + ww * DecodeF32Lds<D>::kPerWave;
      const float f = mw[ww] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[ww] - mmax);
      acc += f * ro[hh * RS + d];
      lacc += f * ro[32 * RS + 32 + hh];
    }
    p.part_o[(pbase + hh) * D + d] = acc;
    if (d == 0) {
      p.part_m[pbase + hh] = mmax;
      p.part_l[pbase + hh] = lacc;
    }
  }
}

// Merge the key ranges: o = sum_s f_s O_s / (Rk sum_s f_s l_s), f_s = 2^(m_s - max m); lse = ln of the total.
// What it takes is a few dependent trips to memory, so a thread takes four elements of up to four ranges in one trip and SL groups of
// threads share the ranges of a (row, head): the launcher takes as many as they need for one trip (above 4 SL ranges, several).
// One element of 8 or 24 ranges a thread and trip / this, decode and merge, us, 24 ranges: 1 x 1500 keys, 16 heads of 128, four rows
// 11.5 / 10.6; 63: 1 x 20 000 26.3 / 15.1; 47: 1 x 6000, 32 heads 17.3 / 11.4; 18: 3 x 9000 19.7 / 15.8; 4: 64 x 8192 108.2 / 107.0;
// dealt by length, with the append: 4 paged sequences of 4096 .. 8192 29.6 / 23.4, 48 of 2048 .. 4096 51.8 / 50.1.
template <int D, typename TO, int SL>
__global__ __launch_bounds__(256) void decode_merge_kernel(DecodeParams p, TO* o, float* lse, float inv_rk) {
  constexpr int LPR = D / 4, SLOTS = 256 / LPR, HB = SLOTS / SL, U = 4;  // lanes per row; (head, group) slots; heads; ranges per trip
  __shared__ f32x4 red_o[SL > 1 ? 256 : 1];
  __shared__ float red_m[SLOTS], red_l[SLOTS];
  const int H = p.H, tid = threadIdx.x, c = tid % LPR, place = tid / LPR, group = place % SL;
  const int h = blockIdx.y * HB + place / SL, h_ld = min(h, H - 1);
  const int b = blockIdx.x / p.lq, qi = blockIdx.x % p.lq;
  int S = p.S, first = b * S;  // the batch entry's ranges
  if (p.slots > 0) {
    const RangePlan plan = plan_ranges(p.kvlen, p.B, p.lk, p.slots, p.round_keys, p.min_keys);
    S = __builtin_amdgcn_readlane(plan.S, b);
    first = __builtin_amdgcn_readlane(plan.first, b);
  }
  float mmax = -INFINITY, lacc = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = group; s0 < S; s0 += U * SL) {  // a running (max, sum, acc) triple carries across the trips
    float ms[U], ls[U];
    f32x4 os[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int s = s0 + q * SL;
      const int64_t idx = ((int64_t)(first + min(s, S - 1)) * p.lq + qi) * H + h_ld;
      ms[q] = p.part_m[idx];
      ls[q] = p.part_l[idx];
      os[q] = *reinterpret_cast<const f32x4*>(p.part_o + idx * D + 4 * c);
      if (s >= S) { ms[q] = -INFINITY; os[q] = f32x4{0.f, 0.f, 0.f, 0.f}; ls[q] = 0.f; }  // an infinity of the last range counts once
    }
    float gmax = mmax;
#pragma unroll
    for (int q = 0; q < U; ++q) gmax = fmaxf(gmax, ms[q]);
    const float carry = mmax == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mmax - gmax);
    acc *= carry;
    lacc *= carry;
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const float f = ms[q] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms[q] - gmax);
      acc += f * os[q];
      lacc += f * ls[q];
    }
    mmax = gmax;
  }
  if constexpr (SL > 1) {
    red_o[tid] = acc;
    if (c == 0) { red_m[place] = mmax; red_l[place] = lacc; }
    __syncthreads();
    if (group != 0) return;
    float ms[SL];
#pragma unroll
    for (int q = 0; q < SL; ++q) { ms[q] = red_m[place + q]; mmax = fmaxf(mmax, ms[q]); }
    acc = f32x4{0.f, 0.f, 0.f, 0.f};
    lacc = 0.f;
#pragma unroll
    for (int q = 0; q < SL; ++q) {
      const float f = ms[q] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms[q] - mmax);
      acc += f * red_o[tid + q * LPR];
      lacc += f * red_l[place + q];
    }
  }
  if (h >= H) return;
  // this call's rows are row0 .. row0 + lq - 1 of the lq_total rows of o and lse
  TO* const out = o + (((int64_t)b * p.lq_total + p.row0 + qi) * H + h) * D + 4 * c;
#pragma unroll
  for (int e = 0; e < 4; ++e) store_from_f32(out + e, acc[e] * inv_rk / lacc);
  if (lse && c == 0) lse[((int64_t)b * H + h) * p.lq_total + p.row0 + qi] = (mmax + __builtin_amdgcn_logf(lacc)) * kLn2;
}

size_t workspace_bytes(int B, int lq, int H, int D, int S) {
  return (size_t)B * lq * S * H * (D + 2) * sizeof(float);
}

// `rows` = {row0, lq_total}: the call serves a->lq query rows that are rows row0 .. of lq_total (a->qa / a->qb point at
// row row0; a->o and a->lse at row 0); a plain call has {0, a->lq}
struct RowWindow { int row0, lq_total; };

// How the keys are split: `S` ranges per batch entry, or (slots > 0) up to `slots` ranges dealt by length
struct KeyRanges {
  int S, slots;
  int count(int B) const { return slots > 0 ? slots : B * S; }
};

template <int RK>
DecodeParams decode_params(const TpaFwdArgs* a, KeyRanges ranges, RowWindow rows) {
  DecodeParams p{};
  p.qa = a->qa; p.qb = a->qb; p.ka = a->ka; p.kb = a->kb; p.va = a->va; p.vb = a->vb;
  float* ws = static_cast<float*>(a->workspace);
  const size_t nm = (size_t)ranges.count(a->B) * a->lq * a->H, no = nm * a->dv;
  p.part_o = ws; p.part_m = ws + no; p.part_l = ws + no + nm;
  p.B = a->B; p.lq = a->lq; p.lk = a->lk; p.H = a->H; p.rq = a->rq;
  p.S = ranges.S; p.slots = ranges.slots;
  // (Rank 2 at head size 64 has any length.  Rank 4 there, us, any length / whole rounds, lengths from half on: 28 x 317 keys, 32 heads, two rows 13.9 / 12.6;
  // 2 x 1519, 64 heads, four rows 14.1 / 12.6; mean of 1092 shapes 1.00 of the time by the sizes alone / 0.98.)
  p.round_keys = a->dv == 128 || RK > 2 ? kWaves * kRowsPerBlock / (float)RK : 0.f;
  p.min_keys = (float)least_keys(RK);
  p.kvlen = a->kv_lengths;
  p.climit = a->causal ? causal_offset_of(a) + 1 + rows.row0 : a->lk;
  p.cbr = a->causal == TPA_CAUSAL_BOTTOM_RIGHT;
  p.row0 = rows.row0; p.lq_total = rows.lq_total;
  p.page_table = a->page_table; p.page_size = a->page_size; p.pages_per_seq = a->pages_per_seq;
  const int page_rows = a->page_size * RK;
  p.page_shift = page_rows > 0 && (page_rows & (page_rows - 1)) == 0 ? __builtin_ctz(page_rows) : -1;
  p.qscale = a->sm_scale * kLog2e / ((float)a->rq * (float)RK);
  return p;
}

template <int D, typename TO, int SL>
int launch_merge_t(const TpaFwdArgs* a, const DecodeParams& p, float inv_rk, hipStream_t stream) {
  constexpr int HB = 256 / (D / 4) / SL;
  hipLaunchKernelGGL((decode_merge_kernel<D, TO, SL>), dim3(a->B * a->lq, (a->H + HB - 1) / HB), dim3(256), 0, stream, p, static_cast<TO*>(a->o), a->lse, inv_rk);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

template <int D, typename TO>
int launch_merge(const TpaFwdArgs* a, const DecodeParams& p, float inv_rk, hipStream_t stream) {
  const int S = p.slots > 0 ? (p.slots + p.B - 1) / p.B : p.S;  // dealt by length: on average
  if (S <= 4) return launch_merge_t<D, TO, 1>(a, p, inv_rk, stream);
  if (S <= 8) return launch_merge_t<D, TO, 2>(a, p, inv_rk, stream);
  if (S <= 16) return launch_merge_t<D, TO, 4>(a, p, inv_rk, stream);
  return launch_merge_t<D, TO, 8>(a, p, inv_rk, stream);
}

template <int D, int RK, bool PAGED, int NQ, Reads READS, bool SIDE = false>
int launch_decode_t(const TpaFwdArgs* a, KeyRanges ranges, hipStream_t stream, RowWindow rows) {
  const DecodeParams p = decode_params<RK>(a, ranges, rows);
  auto kern = decode_kernel<D, RK, PAGED, NQ, READS, SIDE>;
  static bool configured[kMaxDevices] = {};
  const size_t lds = DecodeLds<D>::bytes(NQ, SIDE);
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), lds); rc != TPA_OK) return rc;
  const int rpw = NQ * (SIDE ? 32 / a->H : 1);
  dim3 grid((ranges.count(a->B) + 7) / 8 * 8 * ((a->lq + rpw - 1) / rpw), (a->H + 31) / 32);
  hipLaunchKernelGGL(kern, grid, dim3(kWaves * 64), lds, stream, p);
  if (hipGetLastError() != hipSuccess) return TPA_ERR_LAUNCH;
  return launch_merge<D, uint16_t>(a, p, 1.f / (float)RK, stream);
}

template <int D, int RK, bool PAGED>
int launch_decode_f32_t(const TpaFwdArgs* a, KeyRanges ranges, hipStream_t stream, RowWindow rows) {
  const DecodeParams p = decode_params<RK>(a, ranges, rows);
  auto kern = decode_f32_kernel<D, RK, PAGED>;
  static bool configured[kMaxDevices] = {};
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), DecodeF32Lds<D>::kBytes); rc != TPA_OK) return rc;
  dim3 grid((ranges.count(a->B) + 7) / 8 * 8 * a->lq, (a->H + 31) / 32);
  hipLaunchKernelGGL(kern, grid, dim3(kWaves * 64), DecodeF32Lds<D>::kBytes, stream, p);
  if (hipGetLastError() != hipSuccess) return TPA_ERR_LAUNCH;
  return launch_merge<D, float>(a, p, 1.f / (float)RK, stream);
}

template <int D, int RK>
int launch_decode_f32(const TpaFwdArgs* a, KeyRanges ranges, hipStream_t stream, RowWindow rows) {
  if (a->page_table) {
    if (a->page_size <= 0 || (a->page_size * RK) % kRowsPerBlock != 0 ||
        (int64_t)a->pages_per_seq * a->page_size < a->lk)
      return TPA_ERR_SHAPE;
    return launch_decode_f32_t<D, RK, true>(a, ranges, stream, rows);
  }
  return launch_decode_f32_t<D, RK, false>(a, ranges, stream, rows);
}

// 8 and 16 heads leave columns of the matrix instructions to other query rows: 32 / H rows then cost what one does, with about the
// registers of one row (two sets of loads in flight).  Decode and merge, us, two rows of one set of columns each / side by side:
// 64 x 8192 keys, 16 heads of 128, four rows 166.7 / 124.0, two rows 101.7 / 100.8 (HBM); rank 8, head size 64, four rows 348 / 245; 8
// heads of 64, 300 x 1000 keys, four rows 85.4 / 43.4; 1 x 8192, head size 128, rank 4, eight rows 24.0 / 17.7; step of 48 paged sequences of 2046 .. 4096 keys, 16 heads of 128, four tokens 91.2 / 75.7.
// Two sets of rows side by side in one workgroup are slower (158.7 at the first shape): one set of loads in flight.
// One row group per cache slice: each byte is used once and the loads are marked non-temporal (the whole call 5.1 -> 5.75 TB/s).
// Several (more query rows than a workgroup serves): the groups' workgroups run side by side on one XCD and the later one is
// meant to find the slice in its L2, so the loads stay ordinary (four rows at the c4 shape: 1022 MB fetched with non-temporal
// loads, 676 MB = the cache once with ordinary ones).  Two head blocks read the same token rows as well; with two rows and from
// rank 4 on that decides (3 x 9000 keys, 64 heads of 64, rank 4: 24.1 us non-temporal, 22.5 ordinary; rank 2 19.1 / 19.2, paged
// 52.0 / 54.3), with one row from rank 16 on (48 x 4096 keys, 64 heads of 64: rank 4 94 / 93, rank 8 180 / 179 - 187, paged
// 140 / 133; 16 380 / 356 and 270 / 250; 32 831 / 700 and 557 / 468; with one block of loads in flight, non-temporal, 798 and 518).
bool far_rows(const TpaFwdArgs* a) {
  for (const TpaFactor* f : {&a->ka, &a->kb, &a->va, &a->vb})
    if (f->stride_r < 0 || f->stride_r > kFarthestRow) return true;
  return false;
}
template <int D, int RK, bool PAGED>
int launch_decode_rows(const TpaFwdArgs* a, KeyRanges ranges, hipStream_t stream, RowWindow rows) {
  if (far_rows(a)) return launch_decode_t<D, RK, PAGED, 2, Reads::kFar>(a, ranges, stream, rows);
  if (a->lq == 1) {
    if constexpr (RK >= 16)
      if (a->H > 32) return launch_decode_t<D, RK, PAGED, 1, Reads::kOrdinary>(a, ranges, stream, rows);
    return launch_decode_t<D, RK, PAGED, 1, Reads::kStreaming>(a, ranges, stream, rows);
  }
  if (a->H == 8 || a->H == 16) {
    if (a->lq <= 32 / a->H) return launch_decode_t<D, RK, PAGED, 1, Reads::kStreaming, true>(a, ranges, stream, rows);
    return launch_decode_t<D, RK, PAGED, 1, Reads::kOrdinary, true>(a, ranges, stream, rows);
  }
  if (a->lq == 2 && (a->H <= 32 || RK < 4)) return launch_decode_t<D, RK, PAGED, 2, Reads::kStreaming>(a, ranges, stream, rows);
  return launch_decode_t<D, RK, PAGED, 2, Reads::kOrdinary>(a, ranges, stream, rows);
}

template <int D, int RK>
int launch_decode(const TpaFwdArgs* a, KeyRanges ranges, hipStream_t stream, RowWindow rows) {
  if (a->page_table) {
    // a block of 32 (token, rank) rows must not straddle pages, and the table must cover lk
    if (a->page_size <= 0 || (a->page_size * RK) % kRowsPerBlock != 0 ||
        (int64_t)a->pages_per_seq * a->page_size < a->lk)
      return TPA_ERR_SHAPE;
    return launch_decode_rows<D, RK, true>(a, ranges, stream, rows);
  }
  return launch_decode_rows<D, RK, false>(a, ranges, stream, rows);
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

// ranges whose partials (at head size 128) the fixed array of tpa_decode_noalloc holds
int noalloc_room(int B, int lq, int H) { return (int)(TPA_DECODE_NOALLOC_SCRATCH_BYTES / workspace_bytes(B, lq, H, 128, 1)); }

// Key ranges per batch entry that the workspace is sized for.  One workgroup per compute unit is resident (the kernel
// keeps two blocks of loads in flight in registers), so there are as many as fill 256 of them.  A wave then has at
// least one block of rank 2; where that would take more partials than four blocks per wave
// and more than the fixed array of tpa_decode_noalloc holds (at head size 128), it has four.
// (One sequence of 1500 keys, 16 heads of 128, with the merge: 17.3 us with 6 ranges of four blocks per wave, 14.1 with
// 12 of two, 12.3 with 24 of one.)
// The fp32 kernel serves one query row per workgroup, launches at least twice the workgroups per range of the bf16 kernel and so
// asks for at most as many ranges (and never more workspace).
int splits_for(int B, int lq, int lk, int H, int rows_per_group) {
  const int64_t groups = (int64_t)B * ((lq + rows_per_group - 1) / rows_per_group) * ((H + 31) / 32);
  if (groups >= 256) return 1;
  const int want = (int)((256 + groups - 1) / groups);
  const int few = std::min(want, (lk + 4 * kMinKeys - 1) / (4 * kMinKeys));
  return std::max({1, few, std::min({want, (lk + kMinKeys - 1) / kMinKeys, noalloc_room(B, lq, H)})});
}
// The bf16 kernel, which is what callers are told to size the workspace for, serves two query rows per workgroup, or four where eight
// heads lie side by side (launch_decode_rows).  Counted as two, these were at most half as many workgroups as compute units: us, 8
// heads, so / counted as four: 20 x 8192 keys, head size 64, four rows 29.4 / 23.1, rank 8 78.5 / 62.5; 50 x 4096, 128, four rows 62.1 /
// 44.9; 3 x 16384, 64, 16 rows 30.8 / 21.2; 6 x 8192 dealt by length 14.8 / 14.4; one sequence is bound by its chain: 1 x 32768, 128,
// three rows 21.1 / 22.0.  The ranges that this adds are no more than the fixed array holds, so that nothing it took is refused.
int default_splits(int B, int lq, int lk, int H, int rows_per_group) {
  const int two = splits_for(B, lq, lk, H, std::min(rows_per_group, 2));
  if (rows_per_group <= 2) return two;
  return std::max(two, std::min(splits_for(B, lq, lk, H, rows_per_group), noalloc_room(B, lq, H)));
}
int rows_per_workgroup(int H) { return H == 8 ? 4 : 2; }

// From rank 4 on a block holds fewer keys than those counts, which go by the sizes alone, have in mind: with them a wave of a short cache
// has RK / 2 blocks to walk, one after the other, while compute units are idle.  So with the room for their partials there are as many
// ranges as leave one block per wave, within the fixed array's size.  us, by the sizes alone / so: rank 8, head size 128, 1 x 700 keys, 16
// heads 15.2 / 10.8, 32 heads 16.2 / 11.6, 3 x 920 16.1 / 11.6, 2 x 3000 17.3 / 15.1, 32 heads, four rows 23.2 / 21.8; rank 4, 1 x 700 12.5 /
// 10.5, 2 x 3000, 32 heads 14.6 / 13.0; fp32, 2 x 2000, 8 heads of 64, rank 8 32.0 / 21.9, 3 x 900, 32 heads of 128 56.3 / 36.8.  (Rank 2, 1 x 670,
// 32 heads, two rows: 13.4, with twice the ranges 13.8.)
int splits_by_rank(int B, int lq, int lk, int H, int D, int rk, int dtype, int rows_per_group) {
  const int by_size = default_splits(B, lq, lk, H, rows_per_group);
  const int64_t groups = (int64_t)B * ((lq + rows_per_group - 1) / rows_per_group) * ((H + 31) / 32);
  const int keys = rk <= kRowsPerBlock && (rk & (rk - 1)) == 0 ? least_keys(rk) : kMinKeys;  // of a rank that the kernels take
  if (keys >= kMinKeys || groups >= 256) return by_size;
  const int want = (int)((256 + groups - 1) / groups);
  return std::max(by_size, std::min({want, (lk + keys - 1) / keys, noalloc_room(B, lq, H), most_by_rank(dtype, D, rk)}));
}
// and within the room that the call brings
int splits_of_call(const TpaFwdArgs* a, int rows_per_group) {
  const size_t room = a->workspace_bytes / workspace_bytes(a->B, a->lq, a->H, a->dv, 1);
  return std::max(default_splits(a->B, a->lq, a->lk, a->H, rows_per_group),
                  (int)std::min<size_t>(room, splits_by_rank(a->B, a->lq, a->lk, a->H, a->dv, a->rk, a->dtype, rows_per_group)));
}

// How a launch splits the keys if the caller leaves it to us, with partials for B * splits_of_call ranges at hand.
// With lengths per batch entry the ranges are dealt by them; otherwise all entries get one count, which fills the chip
// at most once: 288 workgroups take two rounds, the second nearly empty (48 x 4096 keys, 32 heads of 128: 6 ranges each 69.5 us, 5 48.6).
// What some wave has to do is a whole number of blocks, so there are no more ranges than that number needs: the others would only
// be partials to merge (1 x 20 000 keys, 16 heads of 128: 63 ranges of up to ten blocks per wave 34.3 us, fewer 26.3; 3 x 9000, 32 heads
// 22.1 / 19.7).
KeyRanges choose_ranges(const TpaFwdArgs* a, int rows_per_group) {
  const int S = splits_of_call(a, rows_per_group);
  const int per_range = (a->lq + rows_per_group - 1) / rows_per_group * ((a->H + 31) / 32);  // workgroups of one range
  if (a->kv_lengths && a->B <= kMaxPlanEntries)
    return KeyRanges{S, std::min(std::max(a->B, 256 / per_range), a->B * S)};
  const int keys = least_keys(a->rk), most = (a->lk + keys - 1) / keys;
  const int n = std::max(1, (int)std::min<int64_t>(std::min(S, most), 256 / ((int64_t)a->B * per_range)));
  const int64_t blocks = ((int64_t)a->lk * a->rk + kRowsPerBlock - 1) / kRowsPerBlock, rounds = (blocks + kWaves * n - 1) / (kWaves * n);
  return KeyRanges{(int)((blocks + kWaves * rounds - 1) / (kWaves * rounds)), 0};
}

}  // namespace
}  // namespace tpa

extern "C" int32_t tpa_decode_default_splits(int32_t B, int32_t lq, int32_t lk, int32_t H) {
  if (B <= 0 || lq <= 0 || lk <= 0 || H <= 0) return 0;
  return tpa::default_splits(B, lq, lk, H, tpa::rows_per_workgroup(H));
}

extern "C" size_t tpa_decode_workspace_bytes(int32_t B, int32_t lq, int32_t lk, int32_t H, int32_t dv, int32_t num_splits) {
  if (B <= 0 || lq <= 0 || lk <= 0 || H <= 0 || dv <= 0) return 0;
  const int S = num_splits > 0 ? num_splits : tpa::default_splits(B, lq, lk, H, tpa::rows_per_workgroup(H));
  return tpa::workspace_bytes(B, lq, H, dv, S);
}

size_t tpa_decode_rank_bytes(int B, int lq, int lk, int H, int dv, int rk, int dtype) {
  return tpa::workspace_bytes(B, lq, H, dv, tpa::splits_by_rank(B, lq, lk, H, dv, rk, dtype, dtype == TPA_DTYPE_BF16 ? tpa::rows_per_workgroup(H) : 1));
}

extern "C" size_t tpa_decode_call_workspace_bytes(const TpaFwdArgs* a) {
  if (!a || a->B <= 0 || a->lq <= 0 || a->lk <= 0 || a->H <= 0 || a->dv <= 0 || a->rk <= 0) return 0;
  const size_t base = tpa_decode_workspace_bytes(a->B, a->lq, a->lk, a->H, a->dv, a->num_splits);
  return a->num_splits > 0 ? base : std::max(base, tpa_decode_rank_bytes(a->B, a->lq, a->lk, a->H, a->dv, a->rk, a->dtype));
}

int tpa_decode_mfma_supported(const TpaFwdArgs* a) {
  using namespace tpa;
  if (a->dtype != TPA_DTYPE_BF16) return 0;
  if (a->dk != a->dv || (a->dk != 64 && a->dk != 128)) return 0;
  if (a->rk != 1 && a->rk != 2 && a->rk != 4 && a->rk != 8 && a->rk != 16 && a->rk != 32) return 0;
  if (a->H % 8 != 0) return 0;
  if (a->lq > 64) return 0;
  if (a->q_segment_ids || a->kv_segment_ids) return 0;
  // rows (token, rank) must be uniformly strided: stride_l == rk * stride_r
  const TpaFactor* fs[4] = {&a->ka, &a->kb, &a->va, &a->vb};
  for (const TpaFactor* f : fs) {
    if (f->stride_l != (int64_t)a->rk * f->stride_r) return 0;
    if (!aligned16(f->ptr) || f->stride_r % 8 != 0 || f->stride_b % 8 != 0) return 0;
  }
  if (!aligned16(a->qb.ptr) || a->qb.stride_r % 8 != 0 || a->qb.stride_l % 8 != 0 || a->qb.stride_b % 8 != 0) return 0;
  return 1;
}

int tpa_decode_mfma_launch(const TpaFwdArgs* a, hipStream_t stream) { return tpa_decode_mfma_launch_rows(a, stream, 0, a->lq); }

int tpa_decode_mfma_launch_rows(const TpaFwdArgs* a, hipStream_t stream, int row0, int lq_total) {
  using namespace tpa;
  const RowWindow rows{row0, lq_total};
  const int rows_each = far_rows(a) ? 2 : rows_per_workgroup(a->H);  // as launch_decode_rows has it
  const int S = a->num_splits > 0 ? a->num_splits : default_splits(a->B, a->lq, a->lk, a->H, rows_each);
  if (S > 65535 || (int64_t)a->B * S > 2147483647LL) return TPA_ERR_SHAPE;
  const KeyRanges ranges = a->num_splits > 0 ? KeyRanges{S, 0} : choose_ranges(a, rows_each);
  if (!a->workspace || a->workspace_bytes < workspace_bytes(a->B, a->lq, a->H, a->dv, S)) return TPA_ERR_WORKSPACE;
  if (!aligned16(a->workspace)) return TPA_ERR_ALIGN;
  if (a->dk == 128) {
    switch (a->rk) {
      case 1: return launch_decode<128, 1>(a, ranges, stream, rows);
      case 2: return launch_decode<128, 2>(a, ranges, stream, rows);
      case 4: return launch_decode<128, 4>(a, ranges, stream, rows);
      case 8: return launch_decode<128, 8>(a, ranges, stream, rows);
      case 16: return launch_decode<128, 16>(a, ranges, stream, rows);
      default: return launch_decode<128, 32>(a, ranges, stream, rows);
    }
  }
  switch (a->rk) {
    case 1: return launch_decode<64, 1>(a, ranges, stream, rows);
    case 2: return launch_decode<64, 2>(a, ranges, stream, rows);
    case 4: return launch_decode<64, 4>(a, ranges, stream, rows);
    case 8: return launch_decode<64, 8>(a, ranges, stream, rows);
    case 16: return launch_decode<64, 16>(a, ranges, stream, rows);
    default: return launch_decode<64, 32>(a, ranges, stream, rows);
  }
}

int tpa_decode_f32_supported(const TpaFwdArgs* a) {
  using namespace tpa;
  if (a->dtype != TPA_DTYPE_F32) return 0;
  if (a->dk != a->dv || (a->dk != 64 && a->dk != 128)) return 0;
  if (a->rk != 1 && a->rk != 2 && a->rk != 4 && a->rk != 8 && a->rk != 16 && a->rk != 32) return 0;
  if (a->lq > 64) return 0;
  if (a->q_segment_ids || a->kv_segment_ids) return 0;
  // rows (token, rank) must be uniformly strided: stride_l == rk * stride_r; B rows are read as 16-byte vectors
  const TpaFactor* fs[4] = {&a->ka, &a->kb, &a->va, &a->vb};
  for (const TpaFactor* f : fs)
    if (f->stride_l != (int64_t)a->rk * f->stride_r) return 0;
  const TpaFactor* bs[3] = {&a->kb, &a->vb, &a->qb};
  for (const TpaFactor* f : bs)
    if (!aligned16(f->ptr) || f->stride_r % 4 != 0 || f->stride_l % 4 != 0 || f->stride_b % 4 != 0) return 0;
  return 1;
}

int tpa_decode_f32_launch(const TpaFwdArgs* a, hipStream_t stream) { return tpa_decode_f32_launch_rows(a, stream, 0, a->lq); }

int tpa_decode_f32_launch_rows(const TpaFwdArgs* a, hipStream_t stream, int row0, int lq_total) {
  using namespace tpa;
  const RowWindow rows{row0, lq_total};
  const int S = a->num_splits > 0 ? a->num_splits : default_splits(a->B, a->lq, a->lk, a->H, 1);
  if (S > 65535 || (int64_t)a->B * S > 2147483647LL) return TPA_ERR_SHAPE;
  const KeyRanges ranges = a->num_splits > 0 ? KeyRanges{S, 0} : choose_ranges(a, 1);
  if (!a->workspace || a->workspace_bytes < workspace_bytes(a->B, a->lq, a->H, a->dv, S)) return TPA_ERR_WORKSPACE;
  if (!aligned16(a->workspace)) return TPA_ERR_ALIGN;
  if (a->dk == 128) {
    switch (a->rk) {
      case 1: return launch_decode_f32<128, 1>(a, ranges, stream, rows);
      case 2: return launch_decode_f32<128, 2>(a, ranges, stream, rows);
      case 4: return launch_decode_f32<128, 4>(a, ranges, stream, rows);
      case 8: return launch_decode_f32<128, 8>(a, ranges, stream, rows);
      case 16: return launch_decode_f32<128, 16>(a, ranges, stream, rows);
      default: return launch_decode_f32<128, 32>(a, ranges, stream, rows);
    }
  }
  switch (a->rk) {
    case 1: return launch_decode_f32<64, 1>(a, ranges, stream, rows);
    case 2: return launch_decode_f32<64, 2>(a, ranges, stream, rows);
    case 4: return launch_decode_f32<64, 4>(a, ranges, stream, rows);
    case 8: return launch_decode_f32<64, 8>(a, ranges, stream, rows);
    case 16: return launch_decode_f32<64, 16>(a, ranges, stream, rows);
    default: return launch_decode_f32<64, 32>(a, ranges, stream, rows);
  }
}

// ---------------------------------------------------------------------------------------------
// tpa_decode for callers that cannot allocate device memory (code under HIP graph capture, tight
// serving loops): the split partials go to a fixed array in this code object instead of a caller
// workspace.  Every device the library runs on holds its own copy of the array until the process
// ends.  Host code must not use the array's name as an address (in host code the name is a
// stand-in for the symbol, not device memory); the device address is looked up once per device
// and kept.
namespace tpa {
namespace {

static __device__ __align__(256) unsigned char scratch[TPA_DECODE_NOALLOC_SCRATCH_BYTES];

void* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mutex;

// Device address of `scratch` on the current device (looked up on the first call per device).
int scratch_of_current_device(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return TPA_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return TPA_ERR_LAUNCH;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return TPA_OK;
}

}  // namespace
}  // namespace tpa

extern "C" int tpa_decode_noalloc(const TpaFwdArgs* a, void* stream) {
  using namespace tpa;
  const int rc = tpa_validate_fwd_args(a);
  if (rc != TPA_OK) return rc;
  if (a->q_segment_ids) return TPA_ERR_UNSUPPORTED;
  const bool bf16 = tpa_decode_mfma_supported(a), f32 = !bf16 && tpa_decode_f32_supported(a);
  if (a->kernel == TPA_KERNEL_GENERIC || (!bf16 && !f32)) return TPA_ERR_UNSUPPORTED;  // the split-key kernels only
  const int S = a->num_splits > 0 ? a->num_splits : default_splits(a->B, a->lq, a->lk, a->H, bf16 ? rows_per_workgroup(a->H) : 1);
  if (S > 65535 || (int64_t)a->B * S > 2147483647LL) return TPA_ERR_SHAPE;
  if (workspace_bytes(a->B, a->lq, a->H, a->dv, S) > (size_t)TPA_DECODE_NOALLOC_SCRATCH_BYTES) return TPA_ERR_WORKSPACE;  // partials exceed the fixed array
  void* ptr = nullptr;
  if (int rc2 = scratch_of_current_device(&ptr); rc2 != TPA_OK) return rc2;
  // every (batch entry, query row, key range, head) slot that the merge kernel reads is written by
  // the decode kernel of the same call, so nothing of the previous call's contents has to be cleared
  TpaFwdArgs b = *a;
  b.workspace = ptr;
  b.workspace_bytes = workspace_bytes(a->B, a->lq, a->H, a->dv, S);  // as many ranges as tpa_decode has with what it needs
  return bf16 ? tpa_decode_mfma_launch(&b, static_cast<hipStream_t>(stream)) : tpa_decode_f32_launch(&b, static_cast<hipStream_t>(stream));
}
