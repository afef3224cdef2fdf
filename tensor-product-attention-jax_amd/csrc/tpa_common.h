// Shared device/host helpers for the gfx950 TPA kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tpa_abi.h"

namespace tpa {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(8))) unsigned int u32x8;
typedef __attribute__((ext_vector_type(16))) unsigned int u32x16;
typedef __attribute__((ext_vector_type(8))) float f32x8;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// bf16 bit pattern (in the low or high half of a dword) -> fp32
__device__ __forceinline__ float bf16lo_to_f32(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16hi_to_f32(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float bf16bits_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// two fp32 -> packed bf16 pair (round to nearest even), lo in bits 0..15
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  bf16x2 r;
  r[0] = (__bf16)lo;
  r[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, r);
}

template <typename T>
__device__ __forceinline__ float load_as_f32(const T* p);
template <>
__device__ __forceinline__ float load_as_f32<float>(const float* p) {
  return *p;
}
template <>
__device__ __forceinline__ float load_as_f32<uint16_t>(const uint16_t* p) {
  return bf16bits_to_f32(*p);
}

template <typename T>
__device__ __forceinline__ void store_from_f32(T* p, float v);
template <>
__device__ __forceinline__ void store_from_f32<float>(float* p, float v) {
  *p = v;
}
template <>
__device__ __forceinline__ void store_from_f32<uint16_t>(uint16_t* p, float v) {
  __bf16 b = (__bf16)v;
  *p = __builtin_bit_cast(uint16_t, b);
}

// A value that is the same in all lanes of a wave, as a scalar.  The compiler takes whatever is made from threadIdx.x or read
// from LDS for a vector: branches on it mask lanes, and a buffer load whose scalar offset or resource is made from it
// becomes a loop over the lanes' values.
__device__ __forceinline__ int scalar(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Combine a value with the one held by lane ^ 32.  v_permlane32_swap hands every lane both its
// own value and its partner's (which of the two results holds which depends on the half the
// lane is in), so order-independent reductions need no select.
__device__ __forceinline__ float halves_max(float x) {
  uint32_t u = __float_as_uint(x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
  uint32_t u = __float_as_uint(x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Minimum / maximum / sum of an int over the 64 lanes of a wave, all of them active; every lane gets the result.  Rows of 16 lanes
// by DPP, rows and halves by exchanges, in registers throughout (with six exchanges through the LDS a packed call's two reductions stand in front of its first tile).
template <int CTRL>
__device__ __forceinline__ int lanes_of(int x) { return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false); }
template <typename F>
__device__ __forceinline__ int wave_reduce(int x, F f) {
  x = f(x, lanes_of<0xB1>(x));   // quad_perm [1, 0, 3, 2]
  x = f(x, lanes_of<0x4E>(x));   // quad_perm [2, 3, 0, 1]
  x = f(x, lanes_of<0x141>(x));  // row_half_mirror
  x = f(x, lanes_of<0x140>(x));  // row_mirror
  const auto r = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
  x = f((int)r[0], (int)r[1]);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)x, false, false);
  return f((int)h[0], (int)h[1]);
}
__device__ __forceinline__ int wave_min(int x) { return wave_reduce(x, [](int a, int b) { return min(a, b); }); }
__device__ __forceinline__ int wave_max(int x) { return wave_reduce(x, [](int a, int b) { return max(a, b); }); }
__device__ __forceinline__ int wave_sum(int x) { return wave_reduce(x, [](int a, int b) { return a + b; }); }

// Packed sequences (tpa/tpa.py:369-375 compares ids pairwise): an element of `other` can only
// pair with this workgroup's elements if its id lies within [min, max] of the workgroup's own ids
// `mine[0 .. n_mine)`.  id_window returns the first and last such index of other[0 .. n_other) (last = -1 if
// there is none): exact for ids that do not decrease along the sequence, conservative otherwise
// (the per-pair mask still decides).  `red` = 3 ints of LDS per wave; every thread of the workgroup calls.
// It stands before the first tile, so what counts is its way through memory and barriers: every wave finds the range of the
// workgroup's ids by itself, four loads of either side are in flight together, and the waves meet once (with atomics of the waves
// on four words, five barriers and one id per load and lane: backward of 32 768 tokens x 16 heads x 128 in documents of 1558
// 1134 instead of 1059 us, of 2 x 1224 x 64 x 64 102 instead of 99, its forward 43.2 instead of 41.4).
__device__ __forceinline__ void id_range(const int32_t* mine, int n_mine, int32_t& smin, int32_t& smax) {
  smin = INT32_MAX; smax = INT32_MIN;
  for (int base = threadIdx.x & 63; base < n_mine; base += 256) {
    int32_t ids[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) ids[u] = mine[min(base + 64 * u, n_mine - 1)];  // past the end: the last again
#pragma unroll
    for (int u = 0; u < 4; ++u) { smin = min(smin, ids[u]); smax = max(smax, ids[u]); }
  }
  smin = wave_min(smin); smax = wave_max(smax);
}
// first / last index and count over the workgroup's waves, each thread's own going in
template <int NT>
__device__ __forceinline__ void window_of_waves(int32_t* red, int& lo, int& hi, int& cnt) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  lo = wave_min(lo); hi = wave_max(hi); cnt = wave_sum(cnt);
  if (lane == 0) { red[w] = lo; red[NW + w] = hi; red[2 * NW + w] = cnt; }
  __syncthreads();
  const bool one = lane < NW;
  lo = scalar(wave_min(one ? red[lane] : INT32_MAX));
  hi = scalar(wave_max(one ? red[NW + lane] : -1));
  cnt = scalar(wave_sum(one ? red[2 * NW + lane] : 0));
  __syncthreads();  // the tiles reuse this memory
}
// smin, smax = the range of the workgroup's own ids; cnt = elements of `other` inside it.  Four ids per load from the first 16-byte
// boundary on, the up to six around it by one lane each.
template <int NT>
__device__ __forceinline__ void id_window(const int32_t* mine, int n_mine, const int32_t* other, int n_other, int32_t* red,
                                          int tid, int& first, int& last, int& cnt, int32_t& smin, int32_t& smax) {
  n_other = max(n_other, 0);
  const int head = min((int)(-(reinterpret_cast<uintptr_t>(other) >> 2) & 3), n_other), n4 = (n_other - head) & ~3;
  int4 ids[4];
  auto request = [&](int base) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (base + 4 * NT * u < n4) ids[u] = *reinterpret_cast<const int4*>(other + head + base + 4 * NT * u);
  };
  request(4 * tid);  // on their way while the workgroup's own ids are looked at
  const bool edge = tid < n_other - n4;
  const int edge_t = tid < head ? tid : n4 + tid;
  int32_t edge_id = 0;
  if (edge) edge_id = other[edge_t];
  id_range(mine, n_mine, smin, smax);
  first = INT32_MAX, last = -1, cnt = 0;
  auto visit = [&](int t, int32_t sid) __attribute__((always_inline)) {
    if (sid >= smin && sid <= smax) { first = min(first, t); last = max(last, t); ++cnt; }
  };
  if (edge) visit(edge_t, edge_id);
  for (int base = 4 * tid; base < n4; base += 16 * NT) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int at = base + 4 * NT * u, t = head + at;
      if (at < n4) { visit(t, ids[u].x); visit(t + 1, ids[u].y); visit(t + 2, ids[u].z); visit(t + 3, ids[u].w); }
    }
    request(base + 16 * NT);
  }
  window_of_waves<NT>(red, first, last, cnt);
}
template <int NT>
__device__ __forceinline__ void id_window(const int32_t* mine, int n_mine, const int32_t* other, int n_other, int32_t* red,
                                          int tid, int& first, int& last) {
  int cnt;
  int32_t smin, smax;
  id_window<NT>(mine, n_mine, other, n_other, red, tid, first, last, cnt, smin, smax);
}

// The windows of all blocks of `block` rows (keys) of a call, found by the launch that reconstructs the dense arrays: once per batch
// entry and block where the attention kernels found them once per head too, each on its way to its first tile.  us, found by the
// attention kernels / here: training step of 3 x 1777 tokens, 16 heads of 64, documents of 421 115.5 / 110.3; 2 x 13 505 of 284 527 /
// 492; 14 x 569 of 129, rank 8 157.5 / 153.3; 1 x 20 000, 32 heads of 128, of 1000 1806 / 1743; forward alone 2 x 13 505 124 / 113, 14 x 569
// 42.2 / 38.8, 5 x 9865, 16 heads of 128, of 477 472 / 458.
// In short calls of few heads the attention kernels find them in less time than that launch takes longer: us, here / by them, 1 x 58 tokens, 8 heads of
// 64, backward 16.6 / 15.7, 2 x 323 25.8 / 24.9; 1 x 82, rank 8, forward 11.9 / 11.5.  By (batch, head) pairs times tokens, mean of the time by them over the
// time here, 700 shapes: forward to 2048 0.98, to 4096 0.99, to 8192 1.02, to 65 536 1.016, beyond 1.05; backward to 4096 0.975, to 8192 0.99, to 16 384
// 1.01, to 65 536 1.02, beyond 1.03.  `least`: of the forward's and of the backward's;
// from rank 16 on the workgroups of Q, which find them, have done before K and V are made (3 x 40 heads of 128, 24 tokens, forward 12.9 / 14.0; mean of 106 shapes
// below 8192 1.045, of 55 backward 1.015).
inline bool windows_ahead_pay(int B, int H, int lq, int lk, int64_t least) { return (int64_t)B * H * (lq > lk ? lq : lk) >= least; }
struct IdWindow { int32_t first, last, count, least, most; };  // what id_window finds
struct WindowJob {
  const int32_t *mine, *other;  // ids [B, n_mine], [B, n_other]; mine = null: no such job
  const int32_t* other_len;     // [B] elements of `other`, or null (= n_other)
  int n_mine, n_other, block;
  int keys;                     // 0: blocks of rows that look for keys, 1: the other way round
  int causal, coff;             // as the attention kernels have them
  int32_t* out;                 // an IdWindow per batch entry, block and copy; strides in int32
  int64_t stride_b, stride_block, stride_copy;
  int copies;
};
// The elements of `other` that the mask leaves a block: [begin, begin + n)
__device__ __forceinline__ void window_range(const WindowJob& j, int b, int x0, int& begin, int& n) {
  begin = 0;
  const int len = j.other_len ? max(0, min(j.other_len[b], j.n_other)) : j.n_other;
  if (!j.causal) { n = len; return; }
  if (j.keys) {  // rows from the tile of 64 on that holds the first one
    begin = min(max(x0 - j.coff, 0) / 64 * 64, len);
    n = len - begin;
  } else {
    const int coff = j.coff + (j.causal == TPA_CAUSAL_BOTTOM_RIGHT ? len - j.n_mine : 0);
    n = max(0, min(len, min(x0 + j.block, j.n_mine) + coff));
  }
}
// workgroup `at` of `of` workgroups of NT threads that share out the blocks of batch entry b; red: 3 ints of LDS per wave
template <int NT>
__device__ __forceinline__ void find_windows(const WindowJob& j, int b, int at, int of, int32_t* red, int tid) {
  for (int blk = at; blk < (j.n_mine + j.block - 1) / j.block; blk += of) {
    const int x0 = blk * j.block;
    int begin, n;
    window_range(j, b, x0, begin, n);
    IdWindow w;
    id_window<NT>(j.mine + (int64_t)b * j.n_mine + x0, min(j.block, j.n_mine - x0), j.other + (int64_t)b * j.n_other + begin, n, red, tid,
                  w.first, w.last, w.count, w.least, w.most);
    for (int c = tid; c < j.copies; c += NT) *reinterpret_cast<IdWindow*>(j.out + b * j.stride_b + blk * j.stride_block + c * j.stride_copy) = w;
  }
}

// Segment ids inside the window.  A workgroup visits every tile that one of its rows needs, a wave owns 32 of them and often a
// single document, so a wave looks at each tile's 64 ids itself: a tile without an id in the range of its own rows is left out, and
// one that holds nothing but the one id of all of them needs no mask.  Both are exact for any order of the ids.
// Forward and backward of 3 x 1777 bf16 tokens, 16 heads of 64, documents of 421 tokens: 133.7 -> 129.0 us.  The fp32 kernels only leave
// tiles out (the mask is little beside six products): 8 x 2000, 8 heads of 64, of 300 529 -> 492; 2 x 9000 of 2000 1756 -> 1681.
enum { kNoneOfThem = 0, kSomeOfThem = 1, kAllOfThem = 2 };
template <bool SEG, int NB>
struct TileIds {
  int32_t least, most;
  __device__ __forceinline__ explicit TileIds(const int32_t (&own)[NB]) : least(0), most(0) {
    if constexpr (SEG) {
      least = most = own[0];
#pragma unroll
      for (int nb = 1; nb < NB; ++nb) { least = min(least, own[nb]); most = max(most, own[nb]); }
      least = scalar(wave_min(least)); most = scalar(wave_max(most));
    }
  }
  // `tile` = the tile's 64 ids in LDS
  __device__ __forceinline__ int look(const int32_t* tile, int lane) const {
    if constexpr (!SEG) return kAllOfThem;
    const int32_t id = tile[lane];
    if (__ballot(id >= least && id <= most) == 0) return kNoneOfThem;
    return least == most && __ballot(id != least) == 0 ? kAllOfThem : kSomeOfThem;
  }
};

// Which of the eight (block, batch) pairs of round `round` the workgroups on XCD `xcd` take, with
// pair = block_rank * B + batch.  Workgroup ids map to XCDs statically, so with a fixed direction
// one XCD would collect the heaviest causal block of every round; odd rounds therefore reverse the
// order of the blocks.  Where B divides 8 only the block rank is reversed and the batch entry is
// kept, so that an XCD keeps meeting the same batch entries (their K/V factors stay in its L2);
// where B is a multiple of 8 a round holds one block rank only and nothing needs to move.
__device__ __forceinline__ int xcd_pair_slot(int round, int xcd, int B) {
  if (!(round & 1) || B % 8 == 0) return xcd;
  if (8 % B == 0) return (8 / B - 1 - xcd / B) * B + xcd % B;
  return 7 - xcd;
}

// Workgroup id -> (block, batch) pair and head for the kernels whose heads share the pair's B factors: the heads of a
// pair sit on one XCD (workgroup ids are dealt round-robin to the eight) and find the factors in its L2.  With fewer than
// eight pairs, or a number that leaves some XCDs a round more than others, that would idle XCDs - one pair of 64 heads ran
// on 32 of 256 compute units - so the heads then go in `groups` groups that are placed like pairs of their own.
__device__ __forceinline__ bool pair_of_workgroup(int id, int npairs, int H, int B, int groups, int& pair, int& h) {
  const int xcd = id & 7, slot = id >> 3, per_group = H / groups;
  const int round = slot / per_group, x = round * 8 + xcd_pair_slot(round, xcd, B * groups);
  pair = x / groups;
  h = x % groups * per_group + slot % per_group;
  return x < npairs * groups;
}
inline int head_groups(int64_t npairs, int H) {
  if (npairs >= 64) return 1;  // the last round is a small part of the launch
  int groups = 1;
  for (int g = 1; g <= 8 && H % g == 0; g *= 2) {
    groups = g;
    if (npairs * g % 8 == 0) break;
  }
  return groups;
}
inline int64_t workgroups_of(int64_t npairs, int H, int groups) { return (npairs * groups + 7) / 8 * 8 * (H / groups); }

// Workgroup id -> (batch, head) pair and block rank for the kernels over dense arrays, which belong to one pair: an XCD owns whole
// pairs and runs them in `groups` groups, whose sizes differ by one at most; inside a group the blocks go in order of their
// rank, the same block of all its pairs side by side.  False: the XCD has a pair less than the others.
__device__ __forceinline__ bool pair_in_group(int id, int npairs, int groups, int nblk, int& pair, int& rank) {
  const int xcd = id & 7, slot = id >> 3, per_xcd = (npairs + 7) / 8;
  const int small = per_xcd / groups, larger = per_xcd - small * groups;  // pairs of a group; groups that have one more
  const int first_small = larger * (small + 1);
  const bool large = slot < first_small * nblk;
  const int size = large ? small + 1 : small, at = large ? slot : slot - first_small * nblk;
  const int grp = at / (size * nblk), rem = at - grp * size * nblk;
  rank = rem / size;
  pair = ((large ? 0 : first_small) + grp * size + rem - rank * size) * 8 + xcd;
  return pair < npairs;
}
inline int64_t pair_group_workgroups(int npairs, int nblk) { return (int64_t)((npairs + 7) / 8) * nblk * 8; }
// as many groups as come nearest to `size` pairs in each
inline int pair_groups(int npairs, int size) {
  const int per_xcd = (npairs + 7) / 8, n = (2 * per_xcd + size - 1) / (2 * size);
  return n < 1 ? 1 : n;
}

// Causal offset of a forward call as the kernels take it: row i sees keys <= i + offset.  Offsets
// of lk and more mask nothing and offsets of -lq and less mask everything, so the value is clamped
// to that range (keeps the kernels' index arithmetic far from overflow); 0 without the causal mask.
// With TPA_CAUSAL_BOTTOM_RIGHT the forward kernels add (keys of the batch entry - lq) themselves, since
// that differs per entry under kv_lengths; the range is then twice as wide.
inline int clamp_causal_offset(int offset, int lo, int hi) { return offset < lo ? lo : (offset > hi ? hi : offset); }
inline int causal_offset_of(const TpaFwdArgs* a) {
  if (!a->causal) return 0;
  if (a->causal == TPA_CAUSAL_BOTTOM_RIGHT) return clamp_causal_offset(a->causal_offset, -a->lq - a->lk, a->lq + a->lk);
  return clamp_causal_offset(a->causal_offset, -a->lq, a->lk);
}
// keys from here on are behind every query's mask, whatever the lengths of the batch entries
inline int keys_in_reach(const TpaFwdArgs* a) {
  if (a->causal != TPA_CAUSAL_TOP_LEFT) return a->lk;
  const int end = a->lq + causal_offset_of(a);
  return end < 0 ? 0 : end < a->lk ? end : a->lk;
}
// the backward takes no kv_lengths, so bottom-right alignment is the fixed offset lk - lq
inline int causal_offset_of(const TpaBwdArgs* a) {
  if (!a->causal) return 0;
  const int base = a->causal == TPA_CAUSAL_BOTTOM_RIGHT ? a->lk - a->lq : 0;
  return clamp_causal_offset(clamp_causal_offset(a->causal_offset, -a->lq - a->lk, a->lq + a->lk) + base, -a->lq, a->lk);
}

// Raise a kernel's dynamic LDS limit above the 64 KB a kernel gets without asking.  The attribute
// belongs to one device's copy of the code, so it is set once per device (`done` is the calling
// launcher's own table; a race between two first launches only repeats the same call).
constexpr int kMaxDevices = 64;
inline int raise_lds_limit(bool (&done)[kMaxDevices], const void* kern, size_t bytes) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return TPA_ERR_LAUNCH;
  if (dev < kMaxDevices && done[dev]) return TPA_OK;
  if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) return TPA_ERR_LAUNCH;
  if (dev < kMaxDevices) done[dev] = true;
  return TPA_OK;
}

}  // namespace tpa

// host-side entry points of the individual kernel files (launchers return TPA_* codes)
int tpa_validate_fwd_args(const TpaFwdArgs* a);  // the checks every forward entry point makes first
int tpa_generic_launch(const TpaFwdArgs* a, hipStream_t stream);
int mha_generic_launch(const MhaFwdArgs* a, hipStream_t stream);
int tpa_prefill_mfma_supported(const TpaFwdArgs* a);
int tpa_prefill_mfma_launch(const TpaFwdArgs* a, hipStream_t stream);
int mha_prefill_mfma_supported(const MhaFwdArgs* a);
int mha_prefill_mfma_launch(const MhaFwdArgs* a, hipStream_t stream);
int tpa_prefill_f32_supported(const TpaFwdArgs* a);
int tpa_prefill_f32_launch(const TpaFwdArgs* a, hipStream_t stream);
// bytes of workspace with which that runs on dense fp32 Q, K and V (0: it would not)
size_t tpa_prefill_f32_dense_bytes(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D, int64_t rk);
size_t tpa_prefill_f32_call_bytes(const TpaFwdArgs* a);
// dense fp32 Q (times q_scale), K, V of a forward call in one launch; TPA_ERR_UNSUPPORTED where the vectorised kernel does not apply
// (whole groups of 8 heads of 64 or 128, 16-byte rows)
bool tpa_recon_dense_qkv_f32_takes(const TpaFwdArgs* a);
int tpa_recon_dense_qkv_f32(const TpaFwdArgs* a, float* qd, float* kd, float* vd, float q_scale, hipStream_t stream);
int mha_prefill_f32_supported(const MhaFwdArgs* a);
int mha_prefill_f32_launch(const MhaFwdArgs* a, hipStream_t stream);
int tpa_nomat_pairs_supported(const TpaFwdArgs* a);
int tpa_nomat_pairs_launch(const TpaFwdArgs* a, hipStream_t stream);
size_t tpa_decode_rank_bytes(int B, int lq, int lk, int H, int dv, int rk, int dtype);  // of the partials of as many key ranges as the rank has a use for
int tpa_decode_mfma_supported(const TpaFwdArgs* a);
int tpa_decode_mfma_launch(const TpaFwdArgs* a, hipStream_t stream);
int tpa_decode_f32_supported(const TpaFwdArgs* a);
int tpa_decode_f32_launch(const TpaFwdArgs* a, hipStream_t stream);
// the same for a->lq query rows that are rows row0 .. row0 + a->lq - 1 of lq_total: a->qa / a->qb point at row row0,
// a->o / a->lse at row 0 of the full arrays, the causal mask counts rows from row0
int tpa_decode_mfma_launch_rows(const TpaFwdArgs* a, hipStream_t stream, int row0, int lq_total);
int tpa_decode_f32_launch_rows(const TpaFwdArgs* a, hipStream_t stream, int row0, int lq_total);
int mha_decode_supported(const MhaFwdArgs* a);
int mha_decode_launch(const MhaFwdArgs* a, hipStream_t stream);
int tpa_bwd_launch(const TpaBwdArgs* a, hipStream_t stream, int mfma);
int mha_bwd_launch(const MhaBwdArgs* a, hipStream_t stream, int mfma);
int dense_bwd_mfma_supported(int dtype, int dk, int dv, int64_t lq, int64_t lk, int64_t H, float sm_scale, const void* bias);
int dense_bwd_mfma_launch(const void* q, const void* k, const void* v, const void* d_o, const float* lse, const float* delta,
                          const int32_t* qseg, const int32_t* kvseg, float* dq, float* dk, float* dv, int B, int lq, int lk,
                          int H, int D, float sm_scale, int causal, int causal_offset, const int32_t* qwin, const int32_t* kwin, hipStream_t stream);
// rows (keys) per workgroup of that launch
int dense_bwd_mfma_block(int B, int lq, int lk, int H, int D, int causal, int segments);
int dense_bwd_f32_supported(int dtype, int dk, int dv, int64_t lq, int64_t lk, const void* bias);
int dense_bwd_f32_launch(const float* q, const float* k, const float* v, const float* d_o, const float* lse, const float* delta,
                         const int32_t* qseg, const int32_t* kvseg, float* dq, float* dk, float* dv, int B, int lq, int lk,
                         int H, int D, float sm_scale, int causal, int causal_offset, hipStream_t stream);
size_t tpa_bwd_workspace_size(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t dk, int64_t dv);
size_t mha_bwd_workspace_size(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t dk, int64_t dv, int dtype);
size_t tpa_prefill_dense_bytes(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D);
int tpa_prefill_wants_dense(int64_t lq, int64_t lk, int64_t rk);
size_t tpa_prefill_best_bytes(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t D, int64_t rk);
size_t tpa_prefill_call_bytes(const TpaFwdArgs* a);
// dense bf16 X[B, L, H, D] = (scale/R) sum_r a_r (x) b_r from bf16 factors
int tpa_recon_dense_bf16(const TpaFactor* fa, const TpaFactor* fb, uint16_t* out, int B, int L, int H, int D, int R, float scale, hipStream_t stream);
// dense Q (times q_scale), K, V of a forward call in one launch; TPA_ERR_UNSUPPORTED where the vectorised kernel does not apply
// (and the windows of packed documents, see WindowJob)
// whether the bf16 launch below takes these factors (whole groups of 8 heads, 16-byte rows)
bool tpa_recon_dense_qkv_takes(const TpaFwdArgs* a);
int tpa_recon_dense_qkv_bf16(const TpaFwdArgs* a, uint16_t* qd, uint16_t* kd, uint16_t* vd, float q_scale, const tpa::WindowJob& windows, hipStream_t stream);
