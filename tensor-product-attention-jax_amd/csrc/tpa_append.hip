// Producer step of a TPA layer for gfx950: the six rank factors of n new tokens per sequence as
// one matrix product y = x W^T, rotary position embedding on the B factors of Q and K, and the K / V
// factors written straight into the factored cache (contiguous or paged) that the decode and
// prefill kernels read.  The reference has no such step (its tests draw the factors at random,
// tpa/tpa_test.py:86-91); the arithmetic follows arXiv 2501.06425, section 3.
//
// bf16, three kernels by the number of new tokens: tiles of 256 x 256 or 128 x 128 whose quarters belong to four waves for a large
// prefill chunk, tiles of 64 x 64 or 64 x 128 whose contraction is dealt to four waves for an ordinary one, and for a decode
// step and other few tokens a kernel whose workgroups own 16 columns and split the contraction over their waves.  All of them compute with v_mfma_f32_*_bf16, stage the
// fp32 results in LDS, and finish whole 16-byte chunks of eight columns: a chunk lies inside one rank
// row of one factor (H and D are multiples of 8), so the rotation partners (2j, 2j+1) are inside it.
// Any other dtype / shape: one thread per chunk of eight columns, fp32 arithmetic.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "tpa_common.h"

namespace tpa {
namespace {

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

struct AppendParams {
  const void* x;
  const void* w;
  const float* cosv;
  const float* sinv;
  const int32_t* positions;
  const int32_t* kvlen;
  int32_t* new_kvlen;
  TpaFactor qa, qb, ka, kb, va, vb;
  const int32_t* page_table;
  int page_size, pages_per_seq;
  int B, n, K, H, D, rq, rk, cache_len, rope_len;
  int M, N;          // tokens (B * n), output columns
  int seg[7];        // first column of qa, qb, ka, kb, va, vb, and N
};

// Where chunk (token m, columns c0 .. c0 + 7) of y goes: the factor it belongs to, and the address
// of its first element (nullptr = dropped).  `rotate` = the chunk is part of a rotated B factor;
// `j0` = index of its first rotation pair.
template <typename T>
__device__ __forceinline__ T* chunk_destination(const AppendParams& p, int m, int c0, bool& rotate, int& j0, int& pos) {
  int f = 0;
#pragma unroll
  for (int k = 1; k < 6; ++k) f += c0 >= p.seg[k];
  const int width = (f & 1) ? p.D : p.H;         // qa, ka, va have H columns per rank; qb, kb, vb have D
  const int local = c0 - p.seg[f], r = local / width, e = local % width;
  const int b = m / p.n, i = m % p.n;
  const int base_len = p.kvlen ? max(0, min(p.kvlen[b], p.cache_len)) : 0;
  pos = p.positions ? p.positions[(int64_t)b * p.n + i] : base_len + i;
  pos = max(0, min(pos, p.rope_len - 1));
  rotate = f == 1 || f == 3;
  j0 = e >> 1;
  // (selected member by member: a reference into the argument block would force it into memory)
  auto pick = [&](auto get) __attribute__((always_inline)) {
    return f == 0 ? get(p.qa) : f == 1 ? get(p.qb) : f == 2 ? get(p.ka) : f == 3 ? get(p.kb) : f == 4 ? get(p.va) : get(p.vb);
  };
  T* base = static_cast<T*>(const_cast<void*>(pick([](const TpaFactor& x) { return x.ptr; })));
  const int64_t sb = pick([](const TpaFactor& x) { return x.stride_b; });
  const int64_t sl = pick([](const TpaFactor& x) { return x.stride_l; });
  const int64_t sr = pick([](const TpaFactor& x) { return x.stride_r; });
  if (f < 2) return base + b * sb + (int64_t)i * sl + (int64_t)r * sr + e;
  const int t = base_len + i;                    // token index in the sequence's cache
  if (t >= p.cache_len) return nullptr;
  if (p.page_table) {
    const int64_t page = p.page_table[(int64_t)b * p.pages_per_seq + t / p.page_size];
    return base + page * sb + (int64_t)(t % p.page_size) * sl + (int64_t)r * sr + e;
  }
  return base + b * sb + (int64_t)t * sl + (int64_t)r * sr + e;
}

// rotate the four pairs of a chunk in place: (y[2j], y[2j+1]) by the angle (pos, j0 + j)
__device__ __forceinline__ void rotate_chunk(const AppendParams& p, float (&y)[8], int pos, int j0) {
  const int half = p.D / 2;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float c = p.cosv[(int64_t)pos * half + j0 + j], s = p.sinv[(int64_t)pos * half + j0 + j];
    const float a = y[2 * j], bb = y[2 * j + 1];
    y[2 * j] = a * c - bb * s;
    y[2 * j + 1] = bb * c + a * s;
  }
}

__device__ __forceinline__ void store_chunk(uint16_t* dst, const float (&y)[8]) {
  u32x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = pack_bf16(y[2 * j], y[2 * j + 1]);
  *reinterpret_cast<u32x4*>(dst) = v;
}
__device__ __forceinline__ void store_chunk(float* dst, const float (&y)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) dst[j] = y[j];
}

__device__ __forceinline__ void write_new_lengths(const AppendParams& p) {
  if (p.new_kvlen && blockIdx.x == 0 && blockIdx.y == 0)
    for (int b = threadIdx.x; b < p.B; b += blockDim.x) {
      const int base_len = p.kvlen ? max(0, min(p.kvlen[b], p.cache_len)) : 0;
      p.new_kvlen[b] = min(base_len + p.n, p.cache_len);
    }
}

// Workgroup id -> tile of y.  Ids are dealt to the 8 XCDs round robin; each XCD takes an eighth of the tiles, walking along the
// shorter side of the matrix of tiles, so that what its L2 has to fetch of x and W is least.  False: past its share.
// (Whole rows of tiles per XCD left XCDs idle below eight rows and unequal above: 600 tokens x 5120 columns 71 -> 41 us,
// 1200 x 5120 125 -> 73, 4352 x 1600 110 -> 75.)
__device__ __forceinline__ bool tile_of_workgroup(int id, int ntm, int ntn, int& tm, int& tn) {
  const int64_t tiles = (int64_t)ntm * ntn;
  const int xcd = id & 7, t = (int)((tiles * xcd + 7) / 8) + (id >> 3);  // (workgroup 0 always has one)
  if (ntn <= ntm) { tm = t / ntn; tn = t % ntn; }
  else { tn = t / ntm; tm = t % ntm; }
  return t < (int)((tiles * (xcd + 1) + 7) / 8);
}
inline unsigned tile_workgroups(int ntm, int ntn) { return (unsigned)(((int64_t)ntm * ntn + 7) / 8 * 8); }

// ---- bf16, many new tokens (a prefill chunk): 256 tokens x 256 columns of y per workgroup, four waves
// (one per SIMD, 512 registers each: the 256 accumulators sit in AGPRs).  A wave owns 128 tokens x 128
// columns = 4 x 4 blocks of v_mfma_f32_32x32x16_bf16, computed transposed (A = rows of W, B = tokens), so
// that a lane ends up with runs of four consecutive columns of one token.  A k step reads 8 fragments for
// 16 MFMAs (eight waves of 64 x 128 read 6 for 8 and measured the same time as this form).  x and W tiles of 256 rows x 64 k are double buffered
// in LDS (row stride 72 elements), raw buffer loads over the tile's rows only (rows past the end read as
// zeros and are never stored).
// One wave per SIMD has nobody to hide behind, so the order inside an iteration is fixed by hand:
//   k step 0, 1: fragments of the next step requested, 16 MFMAs
//   k step 2:    fragments of step 3 requested, 16 MFMAs with the stores of the next tile between them
//   barrier
//   k step 3:    fragments of the next tile's step 0 requested, 16 MFMAs with the loads of the tile after next
// Epilogue: each wave stages its fp32 tile through its own quarter of the (now free) buffers, 64 tokens x 64
// columns at a time, and finishes 16-byte chunks; everything that depends on the token alone (sequence,
// position, cache row or page) is worked out once per workgroup into a small LDS table, everything that
// depends on the column alone once per lane and piece.
// WB = blocks of 32 per wave and dimension: 4 (the tile described above) or 2 (128 x 128 tiles, a wave owns
// 64 x 64, 4 fragment reads per 4 MFMAs) for chunks too small to fill the chip with the large tiles.
// KS = groups of four waves that share the contraction of one tile.  Up to 256 small tiles leave a compute unit one workgroup, and
// a k step of theirs is shorter than the way of a load from the L2 (0.87 us per step of 0.2 us of matrix work): two groups
// take half of the steps each, side by side in their own buffers, the sums meet in LDS, and loads are two steps ahead
// instead of one.  2048 tokens x 1600 columns, d_model 4096: 56 -> 45.5 us.
constexpr int kGK = 64, kGS = kGK + 8;
constexpr int kGCS = 64 + 4;                          // row stride of a wave's staged fp32 piece
template <int WB, int KS>
struct GemmTile {
  static constexpr int kM = 64 * WB, kN = 64 * WB;    // tokens, columns per workgroup
  static constexpr int kStage = (kM + kN) * kGS;      // elements per buffer
  static constexpr size_t kLds = KS * 2 * kStage * sizeof(uint16_t) + kM * 5 * sizeof(int32_t);
  static_assert(64 * kGCS <= kStage / 4 && kStage % 16 == 0, "a wave's staged piece fits its slice");
};
template <int WB, int KS>
__global__ __launch_bounds__(256 * KS) void append_gemm_kernel(AppendParams p) {
  using Tile = GemmTile<WB, KS>;
  constexpr int kGM = Tile::kM, kGN = Tile::kN, kGStage = Tile::kStage;
  constexpr int kWT = 32 * WB;                        // tokens / columns per wave
  extern __shared__ __attribute__((aligned(16))) uint16_t gsm_all[];
  int32_t* const table = reinterpret_cast<int32_t*>(gsm_all + KS * 2 * kGStage);  // [5][kGM]: pos, b, i, cache row coordinates
  const int grp = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;  // this group of waves
  uint16_t* const gsm = gsm_all + grp * 2 * kGStage;
  const int tid = threadIdx.x & 255, w = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int wm = w >> 1, wn = w & 1;
  const int ntn = (p.N + kGN - 1) / kGN, ntm = (p.M + kGM - 1) / kGM;
  int tm, tn;
  if (!tile_of_workgroup(blockIdx.x, ntm, ntn, tm, tn)) return;
  const int m0 = tm * kGM, n0 = tn * kGN;
  const uint16_t* x = static_cast<const uint16_t*>(p.x);
  const uint16_t* wt = static_cast<const uint16_t*>(p.w);

  if (grp == 0 && tid < kGM) {  // what the epilogue needs to know about a token (one per thread)
    const int m = min(m0 + tid, p.M - 1);
    const int b = m / p.n, ii = m % p.n;
    const int base_len = p.kvlen ? max(0, min(p.kvlen[b], p.cache_len)) : 0;
    int pos = p.positions ? p.positions[(int64_t)b * p.n + ii] : base_len + ii;
    pos = max(0, min(pos, p.rope_len - 1));
    const int t = base_len + ii;
    int ra = b, rb = t;
    if (t >= p.cache_len) { ra = 0; rb = -1; }  // dropped
    else if (p.page_table) { ra = p.page_table[(int64_t)b * p.pages_per_seq + t / p.page_size]; rb = t % p.page_size; }
    table[tid] = pos; table[kGM + tid] = b; table[2 * kGM + tid] = ii; table[3 * kGM + tid] = ra; table[4 * kGM + tid] = rb;
  }

  if (blockIdx.x == 0) write_new_lengths(p);

  // loader: thread -> chunk tid & 7 of rows (tid >> 3) + 32 q of x and of W
  const int lrow = tid >> 3, lc = tid & 7;
  constexpr int kRsrcFlags = 0x00020000;  // raw 32-bit data format
  const __amdgpu_buffer_rsrc_t x_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x + (int64_t)m0 * p.K), 0, min(kGM, p.M - m0) * p.K * 2, kRsrcFlags);
  const __amdgpu_buffer_rsrc_t w_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(wt + (int64_t)n0 * p.K), 0, min(kGN, p.N - n0) * p.K * 2, kRsrcFlags);
  const int voff = (lrow * p.K + 8 * lc) * 2;
  const int nk = p.K / (kGK * KS), kt0 = grp * nk;  // this group's k steps
  constexpr int NLD = 2 * WB;  // 16-byte chunks of x and of W per thread and tile
  constexpr int NSET = KS;     // register sets of loads under way: tile t waits in set t % NSET
  u32x4 xr[NSET][NLD], wr[NSET][NLD];
  auto load = [&](auto set_c, int kt) __attribute__((always_inline)) {  // (tiles past the last repeat it: loaded, stored, never read)
    constexpr int set = decltype(set_c)::value;
    const int k0 = (kt0 + min(kt, nk - 1)) * kGK;
#pragma unroll
    for (int q = 0; q < NLD; ++q) {
      xr[set][q] = __builtin_amdgcn_raw_buffer_load_b128(x_rs, voff, (32 * q * p.K + k0) * 2, 0);
      wr[set][q] = __builtin_amdgcn_raw_buffer_load_b128(w_rs, voff, (32 * q * p.K + k0) * 2, 0);
    }
  };
  auto stage = [&](auto set_c, int buf) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    uint16_t* xs = gsm + buf * kGStage + lrow * kGS + 8 * lc;
#pragma unroll
    for (int q = 0; q < NLD; ++q) {
      *reinterpret_cast<u32x4*>(xs + 32 * q * kGS) = xr[set][q];
      *reinterpret_cast<u32x4*>(xs + (kGM + 32 * q) * kGS) = wr[set][q];
    }
  };
  f32x16 acc[WB][WB];
#pragma unroll
  for (int cb = 0; cb < WB; ++cb)
#pragma unroll
    for (int tb = 0; tb < WB; ++tb)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[cb][tb][v] = 0.f;
  // (a wave whose columns all lie past the end multiplies zeros: with one wave per SIMD nobody would use the time)
  bf16x8 fa[2][WB], fb[2][WB];
  const int frag_x = (kWT * wm + i) * kGS + 8 * g, frag_w = (kGM + kWT * wn + i) * kGS + 8 * g;
  auto read_frags = [&](auto slot_c, int buf, auto ks_c) __attribute__((always_inline)) {
    constexpr int sl = decltype(slot_c)::value, ks = decltype(ks_c)::value;
    const uint16_t* base = gsm + buf * kGStage + 16 * ks;
#pragma unroll
    for (int cb = 0; cb < WB; ++cb) fa[sl][cb] = *reinterpret_cast<const bf16x8*>(base + frag_w + 32 * cb * kGS);
#pragma unroll
    for (int tb = 0; tb < WB; ++tb) fb[sl][tb] = *reinterpret_cast<const bf16x8*>(base + frag_x + 32 * tb * kGS);
  };
  // acc[cb][tb][v] = y[token kWT wm + 32 tb + i][column kWT wn + 32 cb + 8 (v / 4) + 4 g + v % 4]
  auto mfmas = [&](auto slot_c) __attribute__((always_inline)) {
    constexpr int sl = decltype(slot_c)::value;
#pragma unroll
    for (int cb = 0; cb < WB; ++cb)
#pragma unroll
      for (int tb = 0; tb < WB; ++tb) acc[cb][tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[sl][cb], fb[sl][tb], acc[cb][tb], 0, 0, 0);
  };
  load(IC<0>{}, 0);
  stage(IC<0>{}, 0);
  static_for<NSET>([&](auto n) __attribute__((always_inline)) { load(IC<(decltype(n)::value + 1) % NSET>{}, decltype(n)::value + 1); });
  __syncthreads();
  read_frags(IC<0>{}, 0, IC<0>{});
  auto step = [&](int kt, auto set_c) __attribute__((always_inline)) {  // set_c: where tile kt + 1 waits
    const int cur = kt & 1, nxt = cur ^ 1;
    read_frags(IC<1>{}, cur, IC<1>{});
    __builtin_amdgcn_sched_barrier(0);
    mfmas(IC<0>{});
    __builtin_amdgcn_sched_barrier(0);
    read_frags(IC<0>{}, cur, IC<2>{});
    __builtin_amdgcn_sched_barrier(0);
    mfmas(IC<1>{});
    __builtin_amdgcn_sched_barrier(0);
    read_frags(IC<1>{}, cur, IC<3>{});
    __builtin_amdgcn_sched_barrier(0);
    mfmas(IC<0>{});
    stage(set_c, nxt);
#pragma unroll
    for (int n = 0; n < WB * WB; ++n) {  // the tile stores spread behind the MFMAs
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x200, 2 * NLD / (WB * WB), 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    read_frags(IC<0>{}, nxt, IC<0>{});
    __builtin_amdgcn_sched_barrier(0);
    mfmas(IC<1>{});
    load(set_c, kt + 1 + NSET);
#pragma unroll
    for (int n = 0; n < WB * WB; ++n) {  // the tile loads spread behind the MFMAs
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 2 * NLD / (WB * WB), 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (NSET == 1) {
    for (int kt = 0; kt < nk; ++kt) step(kt, IC<0>{});
  } else {
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
      step(kt, IC<1>{});
      step(kt + 1, IC<0>{});
    }
    if (kt < nk) step(kt, IC<1>{});
  }
  __syncthreads();  // every wave has left the loop: the buffers are free
  if constexpr (KS == 2) {  // the second group hands its sums to the first, lane by lane, and is done
    f32x4* const sums = reinterpret_cast<f32x4*>(gsm_all + 2 * kGStage) + tid;
    static_assert(256 * WB * WB * 16 * sizeof(float) <= 2 * kGStage * sizeof(uint16_t), "the sums fit the second group's buffers");
#pragma unroll
    for (int cb = 0; cb < WB; ++cb)
#pragma unroll
      for (int tb = 0; tb < WB; ++tb)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq)
          if (grp == 1) sums[256 * ((cb * WB + tb) * 4 + vq)] = f32x4{acc[cb][tb][4 * vq], acc[cb][tb][4 * vq + 1], acc[cb][tb][4 * vq + 2], acc[cb][tb][4 * vq + 3]};
    __syncthreads();
    if (grp == 1) return;
#pragma unroll
    for (int cb = 0; cb < WB; ++cb)
#pragma unroll
      for (int tb = 0; tb < WB; ++tb)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          const f32x4 add = sums[256 * ((cb * WB + tb) * 4 + vq)];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[cb][tb][4 * vq + e] += add[e];
        }
  }

  // ---- epilogue: pieces of 64 tokens x 64 columns through this wave's quarter of the buffers
  float* const cs = reinterpret_cast<float*>(gsm) + w * (kGStage / 4);
  const int cc = l & 7, trow = l >> 3;
#pragma unroll
  for (int ch = 0; ch < WB / 2; ++ch) {
    const int c0 = n0 + kWT * wn + 64 * ch + 8 * cc;
    const bool col_ok = c0 < p.N;
    // the column's side of the address: factor, rank row, element
    int f = 0;
#pragma unroll
    for (int k = 1; k < 6; ++k) f += c0 >= p.seg[k];
    const int width = (f & 1) ? p.D : p.H;
    const int local = c0 - p.seg[f], r = local / width, e = local % width;
    const bool rotate = f == 1 || f == 3;
    auto pick = [&](auto get) __attribute__((always_inline)) {
      return f == 0 ? get(p.qa) : f == 1 ? get(p.qb) : f == 2 ? get(p.ka) : f == 3 ? get(p.kb) : f == 4 ? get(p.va) : get(p.vb);
    };
    uint16_t* const base = static_cast<uint16_t*>(const_cast<void*>(pick([](const TpaFactor& t) { return t.ptr; }))) +
                           (int64_t)r * pick([](const TpaFactor& t) { return t.stride_r; }) + e;
    const int64_t sb = pick([](const TpaFactor& t) { return t.stride_b; });
    const int64_t sl = pick([](const TpaFactor& t) { return t.stride_l; });
    const int half_d = p.D / 2;
#pragma unroll
    for (int th = 0; th < WB / 2; ++th) {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int cq = 0; cq < 2; ++cq)
#pragma unroll
        for (int tq = 0; tq < 2; ++tq)
#pragma unroll
          for (int vq = 0; vq < 4; ++vq) {
            const f32x16& t = acc[2 * ch + cq][2 * th + tq];
            *reinterpret_cast<f32x4*>(cs + (32 * tq + i) * kGCS + 32 * cq + 8 * vq + 4 * g) = f32x4{t[4 * vq], t[4 * vq + 1], t[4 * vq + 2], t[4 * vq + 3]};
          }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's own writes have landed
      __builtin_amdgcn_wave_barrier();
      if (!col_ok) continue;
      // everything a pass fetches from memory first (row coordinates, angles), then the arithmetic and the stores; nothing is
      // fetched behind a branch (columns that do not rotate read the first angles and leave them), where each of the eight
      // passes waits for its own.  Calls with their attention, us
      // before / now, d_model 4096: 2048 tokens x 1600 columns 281.1 / 279.5, 8000 x 1440 253 / 247, 16 384 x 720 209 / 203, 3264 x 4096 248 / 241.
      int64_t off[8];
      f32x4 c4[8], s4[8];
#pragma unroll
      for (int pass = 0; pass < 8; ++pass) {
        const int tl = kWT * wm + 64 * th + 8 * pass + trow;  // token within the workgroup's tile
        const int32_t* const place = table + (f < 2 ? kGM : 3 * kGM) + tl;
        const int ra = place[0], rb = place[kGM];
        off[pass] = m0 + tl < p.M && rb >= 0 ? ra * sb + rb * sl : -1;
        const int64_t at = rotate ? (int64_t)table[tl] * half_d + (e >> 1) : 0;
        c4[pass] = *reinterpret_cast<const f32x4*>(p.cosv + at);
        s4[pass] = *reinterpret_cast<const f32x4*>(p.sinv + at);
      }
#pragma unroll
      for (int pass = 0; pass < 8; ++pass) {
        const float* src = cs + (8 * pass + trow) * kGCS + 8 * cc;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(src), hi = *reinterpret_cast<const f32x4*>(src + 4);
        float y[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float a0 = y[2 * j], b0 = y[2 * j + 1];
          const float ya = a0 * c4[pass][j] - b0 * s4[pass][j], yb = b0 * c4[pass][j] + a0 * s4[pass][j];
          y[2 * j] = rotate ? ya : a0;
          y[2 * j + 1] = rotate ? yb : b0;
        }
        if (off[pass] >= 0) store_chunk(base + off[pass], y);
      }
    }
  }
}

// ---- bf16, tiles of 64 tokens x 32 CB columns whose contraction is dealt to the four waves: each multiplies the whole tile by 16 of
// the 64 k of a stage, so that every byte of a stage is read from LDS once (a wave that owns a quarter of the tile reads half of
// both operands), and the four parts are added up at the end.  Stages go from memory straight to LDS, into a ring of NS, one barrier
// for each: behind it everyone's share of the next stage has landed and the slot of this one, whose fragments are in
// registers by then, takes the loads of the stage NS further on.  Loads, fragment reads and matrix instructions take turns - a wave that
// has filled the queue of loads stands still, with its matrix unit.
// What bounds it: bytes into the compute unit, of which the L2 delivers 115 to 135 a ns where nothing else is done, 108 with a
// barrier and a read of each; the ring takes in 16 KB in 0.2 us (0.26 with all units at it) and 24 KB in 0.27, for 0.05 and 0.1 of matrix
// work.  Two stages per barrier, deeper rings: the same.  d_model 4096, us with waves that own quarters and stage through
// registers (two or four groups of them sharing the contraction) / now: 300 tokens x 1600 columns 19.2 / 15.3, 600 x 1600 20.9 / 16.9, 693 x 1600
// 28.4 / 22.4, 844 x 2240 30.5 / 24.8; d_model 8192: 269 x 2560 32.3 / 24.0, 1160 x 1280 55 / 39.  (128 x 128 tiles in this way: 2048 x 1600
// alone 38.2 / 34.8, but the attention behind it, which the power limit holds, takes 9 us more: 268 / 276 together.)
template <int CB>
struct StreamTile {
  static constexpr int TB = 2, NS = 4;
  static constexpr int kM = 32 * TB, kN = 32 * CB;    // tokens, columns per workgroup
  static constexpr int kStage = (kM + kN) * 128;      // bytes of a stage: 64 k of the rows of x, then of W
  static constexpr int kPass = 64;                    // columns of the tile that are added up at a time
  static constexpr int kPS = kPass + 4;               // row stride (floats) of a wave's part of them
  static constexpr int kPart = kM * kPS;
  static constexpr int kBuffers = NS * kStage > 16 * kPart ? NS * kStage : 16 * kPart;
  static constexpr size_t kLds = kBuffers + kM * 5 * sizeof(int32_t);
};
template <int CB>
__global__ __launch_bounds__(256) void append_stream_kernel(AppendParams p) {
  using Tile = StreamTile<CB>;
  constexpr int TB = Tile::TB, NS = Tile::NS;
  constexpr int kTM = Tile::kM, kTN = Tile::kN, NL = TB + CB;  // NL: loads and fragments of a wave per stage
  extern __shared__ __attribute__((aligned(1024))) unsigned char stream_mem[];
  int32_t* const table = reinterpret_cast<int32_t*>(stream_mem + Tile::kBuffers);  // [5][kTM]: pos, b, i, cache row coordinates
  const int tid = threadIdx.x, w = scalar(tid >> 6), l = tid & 63, i = l & 31, g = l >> 5;
  const int ntn = (p.N + kTN - 1) / kTN, ntm = (p.M + kTM - 1) / kTM;
  int tm, tn;
  if (!tile_of_workgroup(blockIdx.x, ntm, ntn, tm, tn)) return;
  const int m0 = tm * kTM, n0 = tn * kTN;

  // A load instruction brings 8 rows x 64 k straight to LDS, 16 bytes a lane in lane order: the lane of chunk c of row r fetches
  // chunk c ^ (r / 2 & 7), so that reads of one chunk of 16 rows in a row meet no bank twice.  (Rows past the end read as zeros.)
  typedef uint32_t Resource __attribute__((ext_vector_type(4)));
  auto resource = [&](const void* base, int rows) __attribute__((always_inline)) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(base);
    return Resource{(uint32_t)scalar((int)(uint32_t)at), (uint32_t)scalar((int)((uint32_t)(at >> 32) & 0xffff)), (uint32_t)scalar(rows * p.K * 2), 0x00020000u};
  };
  const Resource x_rs = resource(static_cast<const uint16_t*>(p.x) + (int64_t)m0 * p.K, min(kTM, p.M - m0));
  const Resource w_rs = resource(static_cast<const uint16_t*>(p.w) + (int64_t)n0 * p.K, min(kTN, p.N - n0));
  const int voff = ((l >> 3) * p.K + 8 * ((l & 7) ^ (4 * (w & 1) + (l >> 4)))) * 2;
  const int nk = p.K / 64;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)stream_mem;
  auto load = [&](auto j_c, int kt, int slot) __attribute__((always_inline)) {  // (stages past the last repeat it: loaded, never used)
    constexpr int j = decltype(j_c)::value;
    const int row = 8 * (4 * j + w - (j < TB ? 0 : 4 * TB));
    const int soff = scalar((row * p.K + 64 * min(kt, nk - 1)) * 2);
    const uint32_t to = (uint32_t)scalar((int)(lds0 + slot * Tile::kStage + 1024 * (4 * j + w)));
    const Resource rs = j < TB ? x_rs : w_rs;
    const int at = voff;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(to), "v"(at), "s"(rs), "s"(soff) : "memory");
  };
  for (int c = 0; c < NS; ++c) static_for<NL>([&](auto j) __attribute__((always_inline)) { load(j, c, c); });

  if (tid < kTM) {  // what the end needs to know about a token (one per thread)
    const int m = min(m0 + tid, p.M - 1);
    const int b = m / p.n, ii = m % p.n;
    const int base_len = p.kvlen ? max(0, min(p.kvlen[b], p.cache_len)) : 0;
    int pos = p.positions ? p.positions[(int64_t)b * p.n + ii] : base_len + ii;
    pos = max(0, min(pos, p.rope_len - 1));
    const int t = base_len + ii;
    int ra = b, rb = t;
    if (t >= p.cache_len) { ra = 0; rb = -1; }  // dropped
    else if (p.page_table) { ra = p.page_table[(int64_t)b * p.pages_per_seq + t / p.page_size]; rb = t % p.page_size; }
    table[tid] = pos; table[kTM + tid] = b; table[2 * kTM + tid] = ii; table[3 * kTM + tid] = ra; table[4 * kTM + tid] = rb;
  }
  if (blockIdx.x == 0) write_new_lengths(p);

  f32x16 acc[CB][TB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[cb][tb][v] = 0.f;
  bf16x8 frag[2][NL];  // TB of x, CB of W
  const unsigned char* const mine = stream_mem + i * 128 + (((2 * w + g) ^ (i >> 1 & 7)) * 16);
  auto read = [&](auto set_c, auto j_c, int slot) __attribute__((always_inline)) {
    constexpr int j = decltype(j_c)::value;
    frag[decltype(set_c)::value][j] = *reinterpret_cast<const bf16x8*>(mine + slot * Tile::kStage + 4096 * j);
  };
  // acc[cb][tb][v] = part of y[token 32 tb + i][column 32 cb + 8 (v / 4) + 4 g + v % 4]
  int slot = 0;
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * NL) : "memory");
  static_for<NL>([&](auto j) __attribute__((always_inline)) { read(IC<0>{}, j, 0); });
  auto step = [&](int kt, auto set_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    const int next = slot + 1 == NS ? 0 : slot + 1;
    // this wave's loads of the next stage have landed and its fragments of this one are here; behind the barrier, everyone's
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * NL) : "memory");
    constexpr int MF = TB * CB;
    static_for<MF>([&](auto n_c) __attribute__((always_inline)) {
      constexpr int n = decltype(n_c)::value;
      constexpr int cb = n / TB, tb = n % TB;
      acc[cb][tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag[set][TB + cb], frag[set][tb], acc[cb][tb], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      static_for<2 * NL>([&](auto e_c) __attribute__((always_inline)) {
        constexpr int e = decltype(e_c)::value;
        if constexpr (e * MF / (2 * NL) == n) {
          if constexpr (e % 2 == 1) read(IC<1 - set>{}, IC<e / 2>{}, next);
          else load(IC<e / 2>{}, kt + NS, slot);
          __builtin_amdgcn_sched_barrier(0);
        }
      });
    });
    slot = next;
  };
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) { step(kt, IC<0>{}); step(kt + 1, IC<1>{}); }
  if (kt < nk) step(kt, IC<0>{});
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // nothing is on its way to the buffers any more, and nobody reads them

  // ---- the four parts of a piece of the tile meet in LDS, and each thread finishes two chunks of eight columns
  constexpr int kPass = Tile::kPass, kPS = Tile::kPS, kCpr = kPass / 8;
  float* const parts = reinterpret_cast<float*>(stream_mem);
  const int cc = tid % kCpr, row0 = tid / kCpr, half_d = p.D / 2;
  static_for<kTN / kPass>([&](auto pass_c) __attribute__((always_inline)) {
    constexpr int pass = decltype(pass_c)::value;
#pragma unroll
    for (int cq = 0; cq < kPass / 32; ++cq)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          const f32x16& t = acc[pass * (kPass / 32) + cq][tb];
          *reinterpret_cast<f32x4*>(parts + w * Tile::kPart + (32 * tb + i) * kPS + 32 * cq + 8 * vq + 4 * g) = f32x4{t[4 * vq], t[4 * vq + 1], t[4 * vq + 2], t[4 * vq + 3]};
        }
    const int c0 = n0 + kPass * pass + 8 * cc;
    int f = 0;
#pragma unroll
    for (int k = 1; k < 6; ++k) f += c0 >= p.seg[k];
    const int width = (f & 1) ? p.D : p.H;
    const int local = c0 - p.seg[f], r = local / width, e = local % width;
    const bool rotate = f == 1 || f == 3;
    auto pick = [&](auto get) __attribute__((always_inline)) {
      return f == 0 ? get(p.qa) : f == 1 ? get(p.qb) : f == 2 ? get(p.ka) : f == 3 ? get(p.kb) : f == 4 ? get(p.va) : get(p.vb);
    };
    uint16_t* const base = static_cast<uint16_t*>(const_cast<void*>(pick([](const TpaFactor& t) { return t.ptr; }))) +
                           (int64_t)r * pick([](const TpaFactor& t) { return t.stride_r; }) + e;
    const int64_t sb = pick([](const TpaFactor& t) { return t.stride_b; }), sl = pick([](const TpaFactor& t) { return t.stride_l; });
    typedef f32x4 Angles __attribute__((aligned(4)));  // the tables may start at any element
    int64_t off[2];
    f32x4 c4[2], s4[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int tl = row0 + u * (256 / kCpr);
      const int32_t* const place = table + (f < 2 ? kTM : 3 * kTM) + tl;
      const int ra = place[0], rb = place[kTM];
      off[u] = c0 < p.N && m0 + tl < p.M && rb >= 0 ? ra * sb + rb * sl : -1;
      const int64_t at = rotate && c0 < p.N ? (int64_t)table[tl] * half_d + (e >> 1) : 0;
      c4[u] = *reinterpret_cast<const Angles*>(p.cosv + at);
      s4[u] = *reinterpret_cast<const Angles*>(p.sinv + at);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float* const src = parts + (row0 + u * (256 / kCpr)) * kPS + 8 * cc;
      f32x4 lo = *reinterpret_cast<const f32x4*>(src), hi = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
      for (int ww = 1; ww < 4; ++ww) {
        lo += *reinterpret_cast<const f32x4*>(src + ww * Tile::kPart);
        hi += *reinterpret_cast<const f32x4*>(src + ww * Tile::kPart + 4);
      }
      float y[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a0 = y[2 * j], b0 = y[2 * j + 1];
        const float ya = a0 * c4[u][j] - b0 * s4[u][j], yb = b0 * c4[u][j] + a0 * s4[u][j];
        y[2 * j] = rotate ? ya : a0;
        y[2 * j + 1] = rotate ? yb : b0;
      }
      if (off[u] >= 0) store_chunk(base + off[u], y);
    }
    __syncthreads();
  });
}

// ---- bf16, few tokens (a decode step): the call is one read of W, and tiles of 64 columns would leave most of the chip idle.
// A workgroup owns 16 columns, up to 64 tokens and all of k: each of its eight waves takes an eighth of the chunks of 64 k, stages
// its own chunk (16 rows of W and the tokens' rows, whole cache lines in 16-byte pieces, kept in flight in registers several
// chunks ahead) in LDS of its own, swizzled, and multiplies it with v_mfma_f32_16x16x32_bf16 - no barrier before the end,
// where a ninth wave, which has looked up destinations and angles meanwhile, adds the eight partial tiles and stores.
// What bounds it: bytes through the compute unit, 128 KB of W (d_model 4096) and 8 KB per token, at some 40 bytes a clock
// behind the first one's way from HBM; hence the tokens are dealt to more workgroups while there are idle ones.
// (Until now operands were read as fragments, half a cache line per row, and the contraction was split over workgroups with
// a second kernel to add the parts.  d_model 4096, us before / now: 1 token x 1600 columns 10.9 / 7.2, 24 x 1440 11.6 / 7.6,
// 48 x 1600 13.5 / 9.5, 64 x 4096 23.5 / 15.3.)
template <int MB>
struct RowsTile {
  static constexpr int kTok = 16 * MB;
  static constexpr int kRows = 16 + kTok;           // staged rows: 16 of W, then the tokens
  static constexpr int kStage = kRows * 64;         // elements of a wave's stage, one chunk of 64 k
  static constexpr int kPS = 20;                    // row stride (floats) of the partial tile, which reuses the stage
  static constexpr int NLD = kRows / 8;             // load instructions of a chunk: 8 rows x 128 bytes each
  static constexpr int NSET = MB >= 4 ? 2 : MB == 2 ? 4 : 6;  // chunks in flight in registers
  static_assert(kTok * kPS * 4 <= kStage * 2, "the partial tile fits the stage");
};
constexpr int kRowWaves = 8;
template <int MB>
__global__ __launch_bounds__((kRowWaves + 1) * 64) void append_rows_kernel(AppendParams p, int nct, int ntb) {
  typedef RowsTile<MB> T;
  constexpr int NLD = T::NLD, NSET = T::NSET;
  extern __shared__ __attribute__((aligned(16))) uint16_t stage_mem[];  // [kRowWaves][kStage]
  const int tid = threadIdx.x, w = scalar(tid >> 6), l = tid & 63;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int ct = slot / ntb * 8 + xcd, tb = slot % ntb;
  if (ct >= nct) return;  // the grid is rounded up to whole groups of 8 column blocks
  const int n0 = 16 * ct, m0 = T::kTok * tb;
  if (w < kRowWaves) {
    const int nchunks = p.K / 64, lrow = l >> 3, lc = l & 7;
    // buffer loads: the resource ends with the last row of the block that exists, rows past it read as zero
    constexpr int kRsrcFlags = 0x00020000;  // raw 32-bit data format
    const __amdgpu_buffer_rsrc_t w_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(static_cast<const uint16_t*>(p.w) + (int64_t)n0 * p.K), 0, min(16, p.N - n0) * p.K * 2, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t x_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(static_cast<const uint16_t*>(p.x) + (int64_t)m0 * p.K), 0, min(T::kTok, p.M - m0) * p.K * 2, kRsrcFlags);
    const int voff = (lrow * p.K + 8 * lc) * 2;
    uint16_t* const st = stage_mem + w * T::kStage;
    u32x4 in[NSET][NLD];
    auto load = [&](auto set_c, int chunk) __attribute__((always_inline)) {
      constexpr int set = decltype(set_c)::value;
#pragma unroll
      for (int q = 0; q < NLD; ++q)
        in[set][q] = __builtin_amdgcn_raw_buffer_load_b128(q < 2 ? w_rs : x_rs, voff, ((q < 2 ? q : q - 2) * 8 * p.K + 64 * chunk) * 2, 0);
    };
    f32x4 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int r16 = l & 15, kg = l >> 4;
    auto take = [&](auto set_c) __attribute__((always_inline)) {
      constexpr int set = decltype(set_c)::value;
#pragma unroll
      for (int q = 0; q < NLD; ++q) *reinterpret_cast<u32x4*>(st + (8 * q + lrow) * 64 + 8 * (lc ^ lrow)) = in[set][q];
    };
    // Each chunk is summed by itself and then added: a chain of matrix instructions over all of a wave's chunks rounds against
    // the whole sum every time (d_model 4096 / 16 384, 48 tokens: 1.6e-4 / 3.2e-4 of the results missed the rounding of the exact
    // sum, 1.2e-4 / 1.7e-4 so; 200 tokens x 1600 columns 19.0 / 19.9 us).
    auto multiply = [&]() __attribute__((always_inline)) {
      f32x4 part[MB];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int at = r16 * 64 + 8 * ((4 * ks + kg) ^ (r16 & 7));
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(st + at);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          part[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(st + (16 + 16 * mb) * 64 + at), b, ks ? part[mb] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[mb] += part[mb];
    };
    const int first = w * nchunks / kRowWaves, end = (w + 1) * nchunks / kRowWaves;  // this wave's chunks
    static_for<NSET>([&](auto n) __attribute__((always_inline)) {
      if (first + decltype(n)::value < end) load(n, first + decltype(n)::value);
    });
    for (int c0 = first; c0 < end; c0 += NSET)
      static_for<NSET>([&](auto n) __attribute__((always_inline)) {
        const int c = c0 + decltype(n)::value;
        if (c < end) {
          take(n);
          if (c + NSET < end) load(n, c + NSET);
          multiply();
        }
      });
    // acc[mb][v] = partial y[token m0 + 16 mb + 4 kg + v][column n0 + r16]
    float* const part = reinterpret_cast<float*>(st);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int v = 0; v < 4; ++v) part[(16 * mb + 4 * kg + v) * T::kPS + r16] = acc[mb][v];
    __syncthreads();
    if (blockIdx.x == 0 && w == 0 && p.new_kvlen)
      for (int b = l; b < p.B; b += 64) p.new_kvlen[b] = min((p.kvlen ? max(0, min(p.kvlen[b], p.cache_len)) : 0) + p.n, p.cache_len);
    return;
  }
  // the last wave looks up where the results go and their angles while the others multiply, then adds and stores
  constexpr int NC = (2 * T::kTok + 63) / 64;  // chunks of eight columns per lane
  uint16_t* dst[NC];
  float cs[NC][4], sn[NC][4];
  bool rotate[NC];
#pragma unroll
  for (int u = 0; u < NC; ++u) {
    const int t = (64 * u + l) >> 1, c0 = n0 + 8 * (l & 1);
    const bool live = t < T::kTok && m0 + t < p.M && c0 < p.N;
    int j0 = 0, pos = 0;
    dst[u] = nullptr;
    rotate[u] = false;
    if (live) dst[u] = chunk_destination<uint16_t>(p, m0 + t, c0, rotate[u], j0, pos);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      cs[u][j] = rotate[u] ? p.cosv[(int64_t)pos * (p.D / 2) + j0 + j] : 1.f;
      sn[u][j] = rotate[u] ? p.sinv[(int64_t)pos * (p.D / 2) + j0 + j] : 0.f;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NC; ++u) {
    if (!dst[u]) continue;
    const int t = (64 * u + l) >> 1;
    f32x4 lo[kRowWaves], hi[kRowWaves];
#pragma unroll
    for (int ww = 0; ww < kRowWaves; ++ww) {
      const float* const src = reinterpret_cast<const float*>(stage_mem + ww * T::kStage) + t * T::kPS + 8 * (l & 1);
      lo[ww] = *reinterpret_cast<const f32x4*>(src);
      hi[ww] = *reinterpret_cast<const f32x4*>(src + 4);
    }
#pragma unroll
    for (int n = 1; n < kRowWaves; n *= 2)
#pragma unroll
      for (int ww = 0; ww < kRowWaves; ww += 2 * n) { lo[ww] += lo[ww + n]; hi[ww] += hi[ww + n]; }
    float y[8] = {lo[0][0], lo[0][1], lo[0][2], lo[0][3], hi[0][0], hi[0][1], hi[0][2], hi[0][3]};
    if (rotate[u]) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = y[2 * j], b = y[2 * j + 1];
        y[2 * j] = a * cs[u][j] - b * sn[u][j];
        y[2 * j + 1] = b * cs[u][j] + a * sn[u][j];
      }
    }
    store_chunk(dst[u], y);
  }
}

// ---- any dtype and shape: one thread per chunk of eight columns
template <typename T>
__global__ __launch_bounds__(256) void append_generic_kernel(AppendParams p) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int nchunks = p.N / 8;
  if (idx < (int64_t)p.M * nchunks) {
    const int m = (int)(idx / nchunks), c0 = 8 * (int)(idx % nchunks);
    const T* xr = static_cast<const T*>(p.x) + (int64_t)m * p.K;
    const T* wr = static_cast<const T*>(p.w) + (int64_t)c0 * p.K;
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = 0.f;
    for (int k = 0; k < p.K; ++k) {
      const float xv = load_as_f32(xr + k);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] += xv * load_as_f32(wr + (int64_t)j * p.K + k);
    }
    bool rotate; int j0, pos;
    T* dst = chunk_destination<T>(p, m, c0, rotate, j0, pos);
    if (dst) {
      if (rotate) rotate_chunk(p, y, pos, j0);
#pragma unroll
      for (int j = 0; j < 8; ++j) store_from_f32(dst + j, y[j]);
    }
  }
  write_new_lengths(p);
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

// The tiles of 256 x 256 and 128 x 128 read the rotation tables four angles at a time, and take what is more than one round of
// the 64 x 64 tiles with two of them on a compute unit (512).  d_model 4096, us of 64 x 64 or 64 x 128 / 128 x 128: 844 tokens x
// 2240 columns (490) 24.8 / 31.3, 2482 x 720 (468) 23.9 / 31.4, 1536 x 1440 (552) 38.3 / 36.4, 600 x 4096 (640) 37.7 / 35.5.
bool gemm_tiles_pay(const AppendParams& p, const TpaAppendArgs* a) {
  const int64_t tiles = (int64_t)((p.M + 63) / 64) * ((p.N + 63) / 64);
  return tiles > 512 && tiles < (1 << 28) && p.K < (1 << 22) && p.D % 8 == 0 && aligned16(a->rope_cos) && aligned16(a->rope_sin);
}

template <int WB, int KS>
int launch_gemm(const AppendParams& p, hipStream_t s) {
  using Tile = GemmTile<WB, KS>;
  constexpr int kM = Tile::kM, kN = Tile::kN;
  const int ntn = (p.N + kN - 1) / kN, ntm = (p.M + kM - 1) / kM;
  auto kern = append_gemm_kernel<WB, KS>;
  static bool configured[kMaxDevices] = {};
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), Tile::kLds); rc != TPA_OK) return rc;
  hipLaunchKernelGGL(kern, dim3(tile_workgroups(ntm, ntn)), dim3(256 * KS), Tile::kLds, s, p);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

template <int CB>
int launch_stream(const AppendParams& p, hipStream_t s) {
  using Tile = StreamTile<CB>;
  const int ntn = (p.N + Tile::kN - 1) / Tile::kN, ntm = (p.M + Tile::kM - 1) / Tile::kM;
  auto kern = append_stream_kernel<CB>;
  static bool configured[kMaxDevices] = {};
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), Tile::kLds); rc != TPA_OK) return rc;
  hipLaunchKernelGGL(kern, dim3(tile_workgroups(ntm, ntn)), dim3(256), Tile::kLds, s, p);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

// What a call of the few-token kernel costs is the bytes that a compute unit takes in: with `mb` blocks of 16 tokens per workgroup,
// rows of W and x of the workgroups that share one, plus as much again as a block for a workgroup's own way.  d_model 4096, us with
// 16 / 32 / 64 tokens per workgroup: 32 tokens x 1600 columns 8.2 / 10.7 / 11.2, 64 x 1600 11.5 / 10.7 / 14.0, 128 x 1600 20 / 16 /
// 13.6, 150 x 800 14.5 / 13.5 / 10.7, 150 x 1440 - / 14.6 / 17.8, 64 x 4096 24 / 19 / 15, 16 x 5120 13.0 / 15.3 / 18.4.
int rows_cost(const AppendParams& p, int mb) {
  const int64_t per_xcd = (int64_t)(((p.N + 15) / 16 + 7) / 8) * ((p.M + 16 * mb - 1) / (16 * mb));
  return (int)std::min<int64_t>((per_xcd + 31) / 32 * (32 + 16 * mb), 1 << 20);
}
// Blocks of 16 tokens per workgroup if the few-token kernel serves the call, 0 if the tiles do, whose time is nearly the same from
// one tile to 100: 12 us at d_model 4096.  us of this kernel / 64 x 64 tiles by cost: d_model 4096, 160 tokens x 720 columns (cost 64)
// 8.3 / 12.2, 128 x 1600 (96) 10.8 / 11.9, 80 x 2240 (128) 13.7 / 12.3, 160 x 1440 (128) 14.0 / 12.0, 128 x 2560 (192) 19.6 / 11.9; 2048, 128 x 1600
// 7.7 / 8.7, 32 x 5120 (128) 11.0 / 8.4; 8192, 128 x 1600 17.2 / 24.4, 146 x 1440 (128) 20.6 / 25.8, 192 x 1600 (192) 30.5 / 24.5.  Cost 128 changes
// sides between 4096 and 5120, where 150 x 1440 takes 15.1 / 17.1 (6144 17.6 / 21.0, 7168 19.4 / 22.8; 3072, 88 x 2560 11.4 / 9.9); from 2048 down to 256
// it is 0.2 - 0.6 slower here, cost 96 between 1.3 faster and the same.
int few_tokens(const AppendParams& p) {
  int mb = 4;
  for (int n : {2, 1})
    if (rows_cost(p, n) < rows_cost(p, mb)) mb = n;
  return rows_cost(p, mb) <= (p.K >= 5120 ? 128 : 96) ? mb : 0;
}

template <int MB>
int launch_rows(const AppendParams& p, hipStream_t s) {
  const int nct = (p.N + 15) / 16, ntb = (p.M + 16 * MB - 1) / (16 * MB);
  const size_t lds = (size_t)kRowWaves * RowsTile<MB>::kStage * sizeof(uint16_t);
  auto kern = append_rows_kernel<MB>;
  static bool configured[kMaxDevices] = {};
  if (int rc = raise_lds_limit(configured, reinterpret_cast<const void*>(kern), lds); rc != TPA_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((nct + 7) / 8 * 8 * ntb), dim3((kRowWaves + 1) * 64), lds, s, p, nct, ntb);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}
bool chunk_ok(const TpaFactor& f) { return aligned16(f.ptr) && f.stride_b % 8 == 0 && f.stride_l % 8 == 0 && f.stride_r % 8 == 0; }

}  // namespace
}  // namespace tpa

// (The size that the decode step's two kernels needed while there were two.)
extern "C" size_t tpa_cache_append_workspace_bytes(int32_t B, int32_t n, int32_t d_model, int32_t H, int32_t D, int32_t rq, int32_t rk, int32_t dtype) {
  if (B <= 0 || n <= 0 || d_model <= 0 || H <= 0 || D <= 0 || rq <= 0 || rk <= 0 || dtype != TPA_DTYPE_BF16) return 0;
  if ((int64_t)B * n > 64 || H % 8 != 0 || D % 8 != 0) return 0;
  for (int slabs = 8; slabs > 1; slabs >>= 1)
    if (d_model % (256 * slabs) == 0) return (size_t)slabs * 64 * (rq + 2 * rk) * (H + D) * sizeof(float);
  return 0;
}

extern "C" int tpa_cache_append(const TpaAppendArgs* a, void* stream) {
  using namespace tpa;
  if (!a) return TPA_ERR_NULL;
  if (a->dtype != TPA_DTYPE_F32 && a->dtype != TPA_DTYPE_BF16) return TPA_ERR_DTYPE;
  if (a->B <= 0 || a->n <= 0 || a->d_model <= 0 || a->H <= 0 || a->D <= 0 || a->rq <= 0 || a->rk <= 0 || a->cache_len <= 0 ||
      a->rope_len <= 0)
    return TPA_ERR_SHAPE;
  // a chunk of eight columns must lie inside one rank row, and rotation pairs must not straddle rows
  if (a->H % 8 != 0 || a->D % 8 != 0) return TPA_ERR_SHAPE;
  if ((int64_t)a->B * a->n > 2147483647LL) return TPA_ERR_SHAPE;
  if (!a->x || !a->w || !a->rope_cos || !a->rope_sin) return TPA_ERR_NULL;
  const TpaFactor* fs[6] = {&a->qa, &a->qb, &a->ka, &a->kb, &a->va, &a->vb};
  for (const TpaFactor* f : fs)
    if (!f->ptr) return TPA_ERR_NULL;
  if (a->new_kv_lengths && a->new_kv_lengths == a->kv_lengths) return TPA_ERR_UNSUPPORTED;
  if (a->page_table && (a->page_size <= 0 || (int64_t)a->pages_per_seq * a->page_size < a->cache_len)) return TPA_ERR_SHAPE;
  if (a->kernel != TPA_KERNEL_AUTO && a->kernel != TPA_KERNEL_GENERIC && a->kernel != TPA_KERNEL_MFMA) return TPA_ERR_UNSUPPORTED;

  AppendParams p{};
  p.x = a->x; p.w = a->w; p.cosv = a->rope_cos; p.sinv = a->rope_sin;
  p.positions = a->positions; p.kvlen = a->kv_lengths; p.new_kvlen = a->new_kv_lengths;
  p.qa = a->qa; p.qb = a->qb; p.ka = a->ka; p.kb = a->kb; p.va = a->va; p.vb = a->vb;
  p.page_table = a->page_table; p.page_size = a->page_size; p.pages_per_seq = a->pages_per_seq;
  p.B = a->B; p.n = a->n; p.K = a->d_model; p.H = a->H; p.D = a->D; p.rq = a->rq; p.rk = a->rk;
  p.cache_len = a->cache_len; p.rope_len = a->rope_len;
  p.M = a->B * a->n;
  const int widths[6] = {a->rq * a->H, a->rq * a->D, a->rk * a->H, a->rk * a->D, a->rk * a->H, a->rk * a->D};
  p.seg[0] = 0;
  for (int k = 0; k < 6; ++k) p.seg[k + 1] = p.seg[k] + widths[k];
  p.N = p.seg[6];

  hipStream_t s = static_cast<hipStream_t>(stream);
  bool mfma = a->kernel != TPA_KERNEL_GENERIC && a->dtype == TPA_DTYPE_BF16 && a->d_model % 64 == 0 && aligned16(a->x) && aligned16(a->w);
  for (const TpaFactor* f : fs) mfma = mfma && chunk_ok(*f);
  if (a->kernel == TPA_KERNEL_MFMA && !mfma) return TPA_ERR_UNSUPPORTED;
  mfma = mfma && p.K < (1 << 24);  // up to 64 rows are read with offsets of 32 bits
  const int few = mfma ? few_tokens(p) : 0;
  if (few) {
    if (const int rc = few == 1 ? launch_rows<1>(p, s) : few == 2 ? launch_rows<2>(p, s) : launch_rows<4>(p, s); rc != TPA_OK) return rc;
  } else if (mfma && gemm_tiles_pay(p, a)) {
    // What counts is the most tiles that a compute unit gets.  One of 256 x 256 takes 14 us and 23 per 1024 of d_model, four of
    // 128 x 128 where a compute unit has as many take 9 and 35: the large ones are ahead where they save a quarter of
    // the small ones, from d_model 1024 on, or the third of three small ones, above 2048.  us, 128 / 256:
    //   d_model 512: 2600 tokens x 5120 columns (4 and 1 tiles) 31.4 / 32.8, 8192 x 5120 (10, 3) 81 / 89, 6600 x 1440 (3, 1) 25.5 / 31.6
    //   1024: 47.7 / 45.0, 134 / 126, 38.3 / 43.9; 2048: 81 / 70, 233 / 206, 64 / 65; 4096: 149 / 121, 439 / 375, 116 / 109
    //   three for two, 4352 x 5120 (6, 2): 2048 133 / 132, 4096 249 / 232, 8192 483 / 434; five for two, 3264 x 5120: 4096 190 / 229
    const int64_t small = (int64_t)((p.M + 127) / 128) * ((p.N + 127) / 128), large = (int64_t)((p.M + 255) / 256) * ((p.N + 255) / 256);
    const int64_t smalls = (small + 255) / 256, larges = (large + 255) / 256;
    // Two groups of waves need an even number of k steps and one tile per compute unit: with their buffers it holds one, with
    // those of one group two.  us with one / two groups: 2048 x 1600 (208 tiles), d_model 4096 56 / 40, 2048 24 / 23, but 512 12.8 / 13.4.
    const int rc = (smalls > 3 * larges ? p.K >= 1024 : smalls == 3 * larges && p.K > 2048) ? launch_gemm<4, 1>(p, s)
                   : p.K % (2 * kGK) == 0 && smalls == 1                                    ? launch_gemm<2, 2>(p, s)
                                                                                            : launch_gemm<2, 1>(p, s);
    if (rc != TPA_OK) return rc;
  } else if (mfma) {
    // One round of 64 x 128 tiles where the 64 x 64 ones would share compute units, us of the latter / the former: d_model 8192, 1160
    // tokens x 1280 columns (380 and 190 of them) 56 / 39, 4096, 844 x 2240 (490, 252) 29.5 / 25.1, 693 x 1600 (275, 143) 25.4 / 22.3; 2048, 1124 x
    // 1280 (360, 180) 15.3 / 15.2; 1024 9.8 / 10.3.
    const int64_t ntm = (p.M + 63) / 64, tiles = ntm * ((p.N + 63) / 64), wide = ntm * ((p.N + 127) / 128);
    if (ntm > 65535 || tiles > 2147483640) return TPA_ERR_SHAPE;
    const int rc = tiles > 256 && wide <= 256 && p.K >= 2048 && p.K < (1 << 22) ? launch_stream<4>(p, s) : launch_stream<2>(p, s);
    if (rc != TPA_OK) return rc;
  } else {
    const int64_t chunks = (int64_t)p.M * (p.N / 8);
    const int64_t blocks = (chunks + 255) / 256;
    if (blocks > 2147483647LL) return TPA_ERR_SHAPE;
    if (a->dtype == TPA_DTYPE_BF16) hipLaunchKernelGGL(append_generic_kernel<uint16_t>, dim3((unsigned)blocks), dim3(256), 0, s, p);
    else hipLaunchKernelGGL(append_generic_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, s, p);
  }
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}
