// Backward pass: gradients of the attention output with respect to the rank factors
// (tpa/tpa.py:168-214,546-995) and, for the dense baseline, with respect to q, k, v
// (tpa/mha.py:40-65).  Any-shape fp32 arithmetic on the vector ALUs, except stages 3 and 4, which
// run on the matrix cores for bf16 inputs with a head size of 64 or 128.
//
// The factored problem is taken through dense intermediates that live in the caller's
// workspace, so that every stage is a plain, separately checkable kernel:
//   1. recon:    Q, K, V [B, l, H, d] = (1/R) sum_r a_r (x) b_r               (tpa/tpa.py:605-606,623)
//   2. delta:    delta[b, h, i] = sum_d o * do, NaN products skipped          (tpa/tpa.py:965-995)
//   3. dq:       one thread per query row walks the keys:  p = exp(x - lse),
//                dp = do . v, ds = scale * p * (dp - delta), dQ += ds * k      (tpa/tpa.py:779-781)
//   4. dkv:      one thread per key walks the query rows: dV += p * do,
//                dK += ds * q                                                  (tpa/tpa.py:765-777)
//   5. project:  da[r, h] = (1/R) sum_d dX[h, d] b[r, d],  db[r, d] = (1/R) sum_h dX[h, d] a[r, h]
//                for X in {Q, K, V}                                            (tpa/tpa.py:767-768,776-777,782-783)
// Rows without a visible key (lse = -inf) contribute nothing (tpa/tpa.py:675-676).
// Gradients are written as fp32 whatever the input type is.
#include <algorithm>

#include "tpa_common.h"

namespace tpa {
namespace {

constexpr int kThreads = 128;  // rows (dq) or keys (dkv) per workgroup
// keys (dq) or rows (dkv) per LDS tile: the tiles of the widest heads stay below 64 KB
constexpr int tile_of(int dmax) { return dmax > 128 ? 16 : 32; }

// ------------------------------------------------------------------------------------ stage 1
template <typename T, typename TO>
__global__ void recon_kernel(TpaFactor fa, TpaFactor fb, TO* out, int L, int H, int D, int R) {
  const int t = blockIdx.x, b = blockIdx.y;
  const T* ap = static_cast<const T*>(fa.ptr) + b * fa.stride_b + t * fa.stride_l;
  const T* bp = static_cast<const T*>(fb.ptr) + b * fb.stride_b + t * fb.stride_l;
  TO* op = out + ((int64_t)b * L + t) * H * D;
  const float inv = 1.f / (float)R;
  for (int idx = threadIdx.x; idx < H * D; idx += blockDim.x) {
    const int h = idx / D, d = idx - h * D;
    float acc = 0.f;
    for (int r = 0; r < R; ++r) acc += load_as_f32(ap + r * fa.stride_r + h) * load_as_f32(bp + r * fb.stride_r + d);
    store_from_f32(op + idx, acc * inv);
  }
}

// bf16 factors -> dense bf16, 8 elements per thread and token.  A workgroup takes kReconTokens
// consecutive tokens and every thread works on the same (head, 16-byte piece) of all of them at
// once, so that several independent load chains are in flight (one token per workgroup left the
// kernel waiting for one small load after the other).  Needs D % 8 == 0 and 16-byte aligned b rows.
constexpr int kReconTokens = 4;
__global__ __launch_bounds__(256) void recon_bf16_kernel(TpaFactor fa, TpaFactor fb, uint16_t* out, int L, int H, int D, int R, float scale) {
  const int t0 = blockIdx.x * kReconTokens, b = blockIdx.y;
  const uint16_t* ap = static_cast<const uint16_t*>(fa.ptr) + b * fa.stride_b;
  const uint16_t* bp = static_cast<const uint16_t*>(fb.ptr) + b * fb.stride_b;
  const float inv = scale / (float)R;
  const int cpr = D / 8;
  for (int idx = threadIdx.x; idx < H * cpr; idx += blockDim.x) {
    const int h = idx / cpr, cc = idx - h * cpr;
    float acc[kReconTokens][8];
#pragma unroll
    for (int u = 0; u < kReconTokens; ++u)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[u][j] = 0.f;
    for (int r = 0; r < R; ++r) {
      float av[kReconTokens];
      u32x4 bv[kReconTokens];
#pragma unroll
      for (int u = 0; u < kReconTokens; ++u) {
        const int64_t t = min(t0 + u, L - 1);
        av[u] = bf16bits_to_f32(ap[t * fa.stride_l + r * fa.stride_r + h]);
        bv[u] = *reinterpret_cast<const u32x4*>(bp + t * fb.stride_l + r * fb.stride_r + 8 * cc);
      }
#pragma unroll
      for (int u = 0; u < kReconTokens; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[u][2 * j] += av[u] * bf16lo_to_f32(bv[u][j]);
          acc[u][2 * j + 1] += av[u] * bf16hi_to_f32(bv[u][j]);
        }
    }
#pragma unroll
    for (int u = 0; u < kReconTokens; ++u) {
      if (t0 + u >= L) break;
      u32x4 pk;
#pragma unroll
      for (int j = 0; j < 4; ++j) pk[j] = pack_bf16(acc[u][2 * j] * inv, acc[u][2 * j + 1] * inv);
      *reinterpret_cast<u32x4*>(out + (((int64_t)b * L + t0 + u) * H + h) * D + 8 * cc) = pk;
    }
  }
}

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
// The same for head counts that are multiples of 8 with 16-byte aligned a rows: a thread owns one
// (token, 16-byte piece of D, group of 8 heads) and reads, per rank, one 16-byte piece of b and
// the 8 head factors as one 16-byte piece of a - 64 multiply-adds per two loads.  Pieces are the
// fastest thread index, so the 16 threads of a (token, head group) store whole rows of D.
// Of the L tokens of a batch entry that lie in `out`, the first `n` are made, and where `lengths` is given no more than lengths[b]: the
// loops over the dense tiles read no key beyond.  A chunk over caches of 8192 tokens, half to wholly full, 4 sequences of 32 heads of
// 128, rank 4, us with all keys made / without: 128 rows 234 / 215, 512 rows 312 / 306; rank 8, 512 rows 328 / 320.
struct ReconJob { TpaFactor fa, fb; void* out; int L, R; float scale; int n; const int32_t* lengths; };
// The backward's delta in the same launch (blockIdx.z = 3): delta[b, h, i] = sum_d o * do, NaN products (an empty row's o)
// skipped; a thread takes the same piece of 8 heads of one row, the sum over d runs across the lanes that share them.
struct DeltaJob { const void *o, *d_o; float* delta; int lq; };
struct ReconJobs { ReconJob job[3]; DeltaJob delta; WindowJob windows[2]; };  // blockIdx.z picks one: several arrays in one launch
template <typename T>
__device__ __forceinline__ void delta_h8(const DeltaJob& j, int64_t t, int g, int cc, int cpr, int b, int H, int D) {
  constexpr int N = 16 / sizeof(T);  // elements of a 16-byte piece
  const bool live = t < j.lq;
  const int64_t at = (((int64_t)b * j.lq + (live ? t : j.lq - 1)) * H + 8 * g) * D + N * cc;
  u32x4 ov[8], gv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    ov[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(static_cast<const T*>(j.o) + at + (int64_t)i * D));
    gv[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(static_cast<const T*>(j.d_o) + at + (int64_t)i * D));
  }
  float mine = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float acc = 0.f;
    auto add = [&](float x) { if (x == x) acc += x; };
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (sizeof(T) == 2) {
        add(bf16lo_to_f32(ov[i][e]) * bf16lo_to_f32(gv[i][e]));
        add(bf16hi_to_f32(ov[i][e]) * bf16hi_to_f32(gv[i][e]));
      } else {
        add(__uint_as_float(ov[i][e]) * __uint_as_float(gv[i][e]));
      }
    }
    acc = dpp_add<0xB1>(acc);
    acc = dpp_add<0x4E>(acc);
    acc = dpp_add<0x141>(acc);
    if (cpr >= 16) acc = dpp_add<0x140>(acc);
    if (cpr == 32) acc += __shfl_xor(acc, 16, 64);
    if (cc == i) mine = acc;
  }
  if (live && cc < 8) j.delta[((int64_t)b * H + 8 * g + cc) * j.lq + t] = mine;
}

// This thread's token t, group g of 8 heads and piece cc of D: shifts where the counts are powers of two (three divisions of 64 bits
// are a microsecond before the first load: 1340 tokens x 16 heads x 128 with the delta 10.6 us, with shifts and its sums by DPP 7.8)
__device__ __forceinline__ void piece_of(int cpr, int hg, int64_t& t, int& g, int& cc, int blk) {
  const int64_t idx = (int64_t)blk * 256 + threadIdx.x;
  if (((cpr & (cpr - 1)) | (hg & (hg - 1))) == 0) {
    const int s = __builtin_ctz(cpr);
    cc = (int)idx & (cpr - 1);
    g = (int)(idx >> s) & (hg - 1);
    t = idx >> (s + __builtin_ctz(hg));
  } else {
    cc = (int)(idx % cpr);
    g = (int)(idx / cpr % hg);
    t = idx / ((int64_t)cpr * hg);
  }
}

__device__ __forceinline__ int tokens_of(int n, const int32_t* lengths, int b) { return lengths ? min(n, lengths[b]) : n; }

// fp32 factors -> dense fp32, in the same way: a thread owns 4 elements of D for 8 heads of a token
__global__ __launch_bounds__(256) void recon_f32_h8_kernel(ReconJobs jobs, int H, int D) {
  const int cpr = D / 4, hg = H / 8;
  int cc, g;
  int64_t t;
  piece_of(cpr, hg, t, g, cc, blockIdx.x);
  const int b = blockIdx.y;
  if (blockIdx.z == 3) return delta_h8<float>(jobs.delta, t, g, cc, cpr, b, H, D);
  const ReconJob job = blockIdx.z == 0 ? jobs.job[0] : blockIdx.z == 1 ? jobs.job[1] : jobs.job[2];
  if (t >= tokens_of(job.n, job.lengths, b)) return;
  const float* ap = static_cast<const float*>(job.fa.ptr) + b * job.fa.stride_b + t * job.fa.stride_l + 8 * g;
  const float* bp = static_cast<const float*>(job.fb.ptr) + b * job.fb.stride_b + t * job.fb.stride_l + 4 * cc;
  f32x4 acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int G = 2;  // ranks whose loads are in flight together
  for (int r0 = 0; r0 < job.R; r0 += G) {
    f32x4 av[G][2], bv[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int r = min(r0 + u, job.R - 1);
      av[u][0] = *reinterpret_cast<const f32x4*>(ap + (int64_t)r * job.fa.stride_r);
      av[u][1] = *reinterpret_cast<const f32x4*>(ap + (int64_t)r * job.fa.stride_r + 4);
      bv[u] = *reinterpret_cast<const f32x4*>(bp + (int64_t)r * job.fb.stride_r);
    }
#pragma unroll
    for (int u = 0; u < G; ++u)
      if (r0 + u < job.R)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += av[u][i / 4][i % 4] * bv[u];
  }
  const float inv = job.scale / (float)job.R;
  float* op = reinterpret_cast<float*>(job.out) + (((int64_t)b * job.L + t) * H + 8 * g) * D + 4 * cc;
#pragma unroll
  for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(op + (int64_t)i * D) = acc[i] * inv;
}

__global__ __launch_bounds__(256) void recon_bf16_h8_kernel(ReconJobs jobs, int H, int D) {
  if (blockIdx.z == 0) {  // the workgroups that start first
    __shared__ int32_t red[3 * 256 / 64];
    if (jobs.windows[0].mine) find_windows<256>(jobs.windows[0], blockIdx.y, blockIdx.x, gridDim.x, red, threadIdx.x);
    if (jobs.windows[1].mine) find_windows<256>(jobs.windows[1], blockIdx.y, gridDim.x - 1 - blockIdx.x, gridDim.x, red, threadIdx.x);
  }
  const TpaFactor fa = blockIdx.z == 0 ? jobs.job[0].fa : blockIdx.z == 1 ? jobs.job[1].fa : jobs.job[2].fa;
  const TpaFactor fb = blockIdx.z == 0 ? jobs.job[0].fb : blockIdx.z == 1 ? jobs.job[1].fb : jobs.job[2].fb;
  uint16_t* const out = static_cast<uint16_t*>(blockIdx.z == 0 ? jobs.job[0].out : blockIdx.z == 1 ? jobs.job[1].out : jobs.job[2].out);
  const int L = blockIdx.z == 0 ? jobs.job[0].L : blockIdx.z == 1 ? jobs.job[1].L : jobs.job[2].L;
  const int R = blockIdx.z == 0 ? jobs.job[0].R : blockIdx.z == 1 ? jobs.job[1].R : jobs.job[2].R;
  const float scale = blockIdx.z == 0 ? jobs.job[0].scale : blockIdx.z == 1 ? jobs.job[1].scale : jobs.job[2].scale;
  const int n = blockIdx.z == 0 ? jobs.job[0].n : blockIdx.z == 1 ? jobs.job[1].n : jobs.job[2].n;
  const int32_t* const lengths = blockIdx.z == 0 ? jobs.job[0].lengths : blockIdx.z == 1 ? jobs.job[1].lengths : jobs.job[2].lengths;
  const int cpr = D / 8, hg = H / 8;
  int cc, g;
  int64_t t;
  piece_of(cpr, hg, t, g, cc, blockIdx.x);
  const int b = blockIdx.y;
  if (blockIdx.z == 3) return delta_h8<uint16_t>(jobs.delta, t, g, cc, cpr, b, H, D);
  if (t >= tokens_of(n, lengths, b)) return;
  const uint16_t* ap = static_cast<const uint16_t*>(fa.ptr) + b * fa.stride_b + t * fa.stride_l + 8 * g;
  const uint16_t* bp = static_cast<const uint16_t*>(fb.ptr) + b * fb.stride_b + t * fb.stride_l + 8 * cc;
  float acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = 0.f;
  // Two ranks per step of the inner product: the head factors of ranks (r, r + 1) and the b elements of the
  // same two ranks are paired into packed bf16 words (16 byte permutes per pair of ranks), and one dot
  // instruction then adds a_r[h] b_r[d] + a_r+1[h] b_r+1[d] to the accumulator - half the instructions of
  // unpacking both and multiplying in fp32, which is what bounds this kernel from rank 8 on.
  constexpr int G = 4;  // ranks whose loads are in flight together (at low ranks the kernel is bound by their latency)
  for (int r0 = 0; r0 < R; r0 += G) {
    u32x4 av[G], bv[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int r = min(r0 + u, R - 1);
      av[u] = *reinterpret_cast<const u32x4*>(ap + (int64_t)r * fa.stride_r);
      bv[u] = *reinterpret_cast<const u32x4*>(bp + (int64_t)r * fb.stride_r);
      if (r0 + u >= R) av[u] = u32x4{0u, 0u, 0u, 0u};  // past the last rank: weight zero
    }
#pragma unroll
    for (int u = 0; u < G; u += 2) {
      if (r0 + u >= R) break;
      uint32_t apair[8], bpair[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        apair[2 * j] = __builtin_amdgcn_perm(av[u + 1][j], av[u][j], 0x05040100u);      // (a_r[2j], a_r+1[2j])
        apair[2 * j + 1] = __builtin_amdgcn_perm(av[u + 1][j], av[u][j], 0x07060302u);  // (a_r[2j+1], a_r+1[2j+1])
        bpair[2 * j] = __builtin_amdgcn_perm(bv[u + 1][j], bv[u][j], 0x05040100u);
        bpair[2 * j + 1] = __builtin_amdgcn_perm(bv[u + 1][j], bv[u][j], 0x07060302u);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          acc[i][j] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, apair[i]), __builtin_bit_cast(bf16x2, bpair[j]), acc[i][j], false);
    }
  }
  const float inv = scale / (float)R;
  uint16_t* op = out + (((int64_t)b * L + t) * H + 8 * g) * D + 8 * cc;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    u32x4 pk;
#pragma unroll
    for (int j = 0; j < 4; ++j) pk[j] = pack_bf16(acc[i][2 * j] * inv, acc[i][2 * j + 1] * inv);
    *reinterpret_cast<u32x4*>(op + (int64_t)i * D) = pk;
  }
}

template <typename T>
__global__ void to_f32_kernel(const T* in, float* out, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = load_as_f32(in + i);
}

// ------------------------------------------------------------------------------------ stage 2
// delta[b, h, i] = sum_d o[b, i, h, d] * do[b, i, h, d], skipping NaN products (an empty row's o).
// Sixteen lanes share a row; with bf16 rows of a multiple of 8 elements each lane takes 16 bytes
// per step, so a wave reads four rows with fully coalesced loads.
template <typename T>
__global__ void delta_kernel(const T* o, const T* d_o, float* delta, int B, int lq, int H, int dv, int vec) {
  const int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;  // over (b, i, h)
  const int sub = threadIdx.x & 15;
  const bool ok = row < (int64_t)B * lq * H;
  float acc = 0.f;
  if (ok) {
    const T* op = o + row * dv;
    const T* gp = d_o + row * dv;
    if constexpr (sizeof(T) == 2) {
      if (vec) {
        for (int d = 8 * sub; d < dv; d += 128) {
          const u32x4 a = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(op + d));
          const u32x4 g = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gp + d));
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float x0 = bf16lo_to_f32(a[j]) * bf16lo_to_f32(g[j]), x1 = bf16hi_to_f32(a[j]) * bf16hi_to_f32(g[j]);
            if (x0 == x0) acc += x0;
            if (x1 == x1) acc += x1;
          }
        }
      }
    }
    if (!(sizeof(T) == 2 && vec)) {
      for (int d = sub; d < dv; d += 16) {
        const float x = load_as_f32(op + d) * load_as_f32(gp + d);
        if (x == x) acc += x;
      }
    }
  }
#pragma unroll
  for (int m = 8; m >= 1; m >>= 1) acc += __shfl_xor(acc, m, 16);
  if (ok && sub == 0) {
    const int h = row % H;
    const int64_t bi = row / H;
    const int i = bi % lq, b = bi / lq;
    delta[((int64_t)b * H + h) * lq + i] = acc;
  }
}

struct DenseParams {
  const float* q;  // [B, lq, H, dk]
  const float* k;  // [B, lk, H, dk]
  const float* v;  // [B, lk, H, dv]
  const void* d_o;  // [B, lq, H, dv], element type T
  const float* lse;    // [B, H, lq]
  const float* delta;  // [B, H, lq]
  const int32_t* qseg;
  const int32_t* kvseg;
  const float* bias;  // [B, lq, lk] or null
  float* dq;          // [B, lq, H, dk]
  float* dk_out;      // [B, lk, H, dk]
  float* dv_out;      // [B, lk, H, dv]
  int B, lq, lk, H, dk, dv;
  float sm_scale;
  int causal;
  int coff;  // with causal: row i sees keys <= i + coff
};

// ------------------------------------------------------------------------------------ stage 3
template <typename T, int DMAX>
__global__ __launch_bounds__(kThreads) void bwd_dq_kernel(DenseParams p) {
  constexpr int kTile = tile_of(DMAX);
  const int b = blockIdx.z, h = blockIdx.y;
  const int row = blockIdx.x * kThreads + threadIdx.x;
  const int dk = p.dk, dv = p.dv;
  extern __shared__ float smem[];
  float* ks = smem;               // [kTile][dk]
  float* vs = smem + kTile * dk;  // [kTile][dv]
  int* segs = reinterpret_cast<int*>(vs + kTile * dv);

  float lse = -INFINITY, delta = 0.f;
  float q[DMAX], g[DMAX], acc[DMAX];
#pragma unroll
  for (int d = 0; d < DMAX; ++d) { q[d] = 0.f; g[d] = 0.f; acc[d] = 0.f; }
  const bool row_ok = row < p.lq;
  if (row_ok) {
    lse = p.lse[((int64_t)b * p.H + h) * p.lq + row];
    delta = p.delta[((int64_t)b * p.H + h) * p.lq + row];
    const float* qp = p.q + (((int64_t)b * p.lq + row) * p.H + h) * dk;
    const T* gp = static_cast<const T*>(p.d_o) + (((int64_t)b * p.lq + row) * p.H + h) * dv;
#pragma unroll
    for (int d = 0; d < DMAX; ++d) {
      if (d < dk) q[d] = qp[d];
      if (d < dv) {
        const float x = load_as_f32(gp + d);
        g[d] = x == x ? x : 0.f;
      }
    }
  }
  const bool live = row_ok && lse > -INFINITY;  // a row without a visible key has no gradient
  const int qseg = (row_ok && p.qseg) ? p.qseg[(int64_t)b * p.lq + row] : 0;

  int k_end = p.lk;
  if (p.causal) k_end = min(p.lk, min(p.lq, (int)(blockIdx.x + 1) * kThreads) + p.coff);
  for (int k0 = 0; k0 < k_end; k0 += kTile) {
    const int nk = min(kTile, k_end - k0);
    __syncthreads();
    for (int idx = threadIdx.x; idx < nk * dk; idx += kThreads) {
      const int t = idx / dk, d = idx - t * dk;
      ks[idx] = p.k[(((int64_t)b * p.lk + k0 + t) * p.H + h) * dk + d];
    }
    for (int idx = threadIdx.x; idx < nk * dv; idx += kThreads) {
      const int t = idx / dv, d = idx - t * dv;
      vs[idx] = p.v[(((int64_t)b * p.lk + k0 + t) * p.H + h) * dv + d];
    }
    if (p.kvseg)
      for (int t = threadIdx.x; t < nk; t += kThreads) segs[t] = p.kvseg[(int64_t)b * p.lk + k0 + t];
    __syncthreads();
    if (!live) continue;
    for (int t = 0; t < nk; ++t) {
      bool keep = true;
      if (p.kvseg) keep = segs[t] == qseg;
      if (p.causal) keep = keep && (k0 + t <= row + p.coff);
      if (!keep) continue;
      float dot = 0.f;
#pragma unroll
      for (int d = 0; d < DMAX; ++d)
        if (d < dk) dot += q[d] * ks[t * dk + d];
      float x = dot * p.sm_scale;
      if (p.bias) x += p.bias[((int64_t)b * p.lq + row) * p.lk + k0 + t];
      const float pt = expf(x - lse);
      float dp = 0.f;
#pragma unroll
      for (int d = 0; d < DMAX; ++d)
        if (d < dv) dp += g[d] * vs[t * dv + d];
      const float ds = p.sm_scale * pt * (dp - delta);
#pragma unroll
      for (int d = 0; d < DMAX; ++d)
        if (d < dk) acc[d] += ds * ks[t * dk + d];
    }
  }
  if (!row_ok) return;
  float* op = p.dq + (((int64_t)b * p.lq + row) * p.H + h) * dk;
#pragma unroll
  for (int d = 0; d < DMAX; ++d)
    if (d < dk) op[d] = acc[d];
}

// ------------------------------------------------------------------------------------ stage 4
template <typename T, int DMAX>
__global__ __launch_bounds__(kThreads) void bwd_dkv_kernel(DenseParams p) {
  constexpr int kTile = tile_of(DMAX);
  const int b = blockIdx.z, h = blockIdx.y;
  const int key = blockIdx.x * kThreads + threadIdx.x;
  const int dk = p.dk, dv = p.dv;
  extern __shared__ float smem[];
  float* qs = smem;                   // [kTile][dk]
  float* gs = smem + kTile * dk;      // [kTile][dv]  upstream gradient rows
  float* ls = gs + kTile * dv;        // [kTile] lse
  float* des = ls + kTile;            // [kTile] delta
  int* segs = reinterpret_cast<int*>(des + kTile);

  float kr[DMAX], vr[DMAX], dkr[DMAX], dvr[DMAX];
#pragma unroll
  for (int d = 0; d < DMAX; ++d) { kr[d] = 0.f; vr[d] = 0.f; dkr[d] = 0.f; dvr[d] = 0.f; }
  const bool key_ok = key < p.lk;
  if (key_ok) {
    const float* kp = p.k + (((int64_t)b * p.lk + key) * p.H + h) * dk;
    const float* vp = p.v + (((int64_t)b * p.lk + key) * p.H + h) * dv;
#pragma unroll
    for (int d = 0; d < DMAX; ++d) {
      if (d < dk) kr[d] = kp[d];
      if (d < dv) vr[d] = vp[d];
    }
  }
  const int kseg = (key_ok && p.kvseg) ? p.kvseg[(int64_t)b * p.lk + key] : 0;

  // under the causal mask only rows at or after this workgroup's first key can see its keys
  const int q_begin = p.causal ? min(p.lq, max((int)blockIdx.x * kThreads - p.coff, 0)) / kTile * kTile : 0;
  for (int q0 = q_begin; q0 < p.lq; q0 += kTile) {
    const int nq = min(kTile, p.lq - q0);
    __syncthreads();
    for (int idx = threadIdx.x; idx < nq * dk; idx += kThreads) {
      const int i = idx / dk, d = idx - i * dk;
      qs[idx] = p.q[(((int64_t)b * p.lq + q0 + i) * p.H + h) * dk + d];
    }
    for (int idx = threadIdx.x; idx < nq * dv; idx += kThreads) {
      const int i = idx / dv, d = idx - i * dv;
      const float x = load_as_f32(static_cast<const T*>(p.d_o) + (((int64_t)b * p.lq + q0 + i) * p.H + h) * dv + d);
      gs[idx] = x == x ? x : 0.f;
    }
    for (int i = threadIdx.x; i < nq; i += kThreads) {
      ls[i] = p.lse[((int64_t)b * p.H + h) * p.lq + q0 + i];
      des[i] = p.delta[((int64_t)b * p.H + h) * p.lq + q0 + i];
      if (p.qseg) segs[i] = p.qseg[(int64_t)b * p.lq + q0 + i];
    }
    __syncthreads();
    if (!key_ok) continue;
    for (int i = 0; i < nq; ++i) {
      const float lse = ls[i];
      bool keep = lse > -INFINITY;
      if (p.qseg) keep = keep && segs[i] == kseg;
      if (p.causal) keep = keep && (key <= q0 + i + p.coff);
      if (!keep) continue;
      float dot = 0.f;
#pragma unroll
      for (int d = 0; d < DMAX; ++d)
        if (d < dk) dot += kr[d] * qs[i * dk + d];
      float x = dot * p.sm_scale;
      if (p.bias) x += p.bias[((int64_t)b * p.lq + q0 + i) * p.lk + key];
      const float pt = expf(x - lse);
      float dp = 0.f;
#pragma unroll
      for (int d = 0; d < DMAX; ++d)
        if (d < dv) {
          const float gd = gs[i * dv + d];
          dp += gd * vr[d];
          dvr[d] += pt * gd;
        }
      const float ds = p.sm_scale * pt * (dp - des[i]);
#pragma unroll
      for (int d = 0; d < DMAX; ++d)
        if (d < dk) dkr[d] += ds * qs[i * dk + d];
    }
  }
  if (!key_ok) return;
  float* okp = p.dk_out + (((int64_t)b * p.lk + key) * p.H + h) * dk;
  float* ovp = p.dv_out + (((int64_t)b * p.lk + key) * p.H + h) * dv;
#pragma unroll
  for (int d = 0; d < DMAX; ++d) {
    if (d < dk) okp[d] = dkr[d];
    if (d < dv) ovp[d] = dvr[d];
  }
}

// ------------------------------------------------------------------------------------ stage 5
// One workgroup (256 threads) per token: da[r, h] and db[r, d] from the token's dense gradient
// dX[h, d].  With STAGE the token's dX (row stride D + 1), a and b sit in LDS; each da output is
// shared by `ns` neighbouring lanes that split the sum over d and combine with lane shuffles.
template <typename T, typename TO, bool STAGE>
__global__ __launch_bounds__(256) void project_kernel(const float* dx, TpaFactor fa, TpaFactor fb, TpaGrad ga, TpaGrad gb, int L, int H,
                                                       int D, int R, int dsh, int nsh) {
  const int t = blockIdx.x, b = blockIdx.y;
  const float* xp = dx + ((int64_t)b * L + t) * H * D;
  const T* ap = static_cast<const T*>(fa.ptr) + b * fa.stride_b + t * fa.stride_l;
  const T* bp = static_cast<const T*>(fb.ptr) + b * fb.stride_b + t * fb.stride_l;
  TO* oa = reinterpret_cast<TO*>(ga.ptr) + b * ga.stride_b + t * ga.stride_l;
  TO* ob = reinterpret_cast<TO*>(gb.ptr) + b * gb.stride_b + t * gb.stride_l;
  const float inv = 1.f / (float)R;
  extern __shared__ __attribute__((aligned(16))) float xs[];  // [H][XS], then b[R][D], then a[R][H]
  if constexpr (STAGE) {
    // D = 1 << dsh here (indices by shifts, not divisions); rows 16 bytes apart in the banks, so
    // that lanes that read 16 bytes of different rows (the da part) spread over the banks
    const int XS = D + 4, d4sh = dsh - 2, d4mask = (D >> 2) - 1;
    float* bs = xs + H * XS;
    float* as = bs + R * D;
    for (int idx = threadIdx.x; idx < (H << d4sh); idx += 256) {
      const int h = idx >> d4sh, d4 = idx & d4mask;
      *reinterpret_cast<f32x4*>(xs + h * XS + 4 * d4) = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(xp + 4 * idx));
    }
    for (int idx = threadIdx.x; idx < (R << dsh); idx += 256) {
      const int r = idx >> dsh, d = idx & (D - 1);
      bs[idx] = load_as_f32(bp + r * fb.stride_r + d);
    }
    for (int idx = threadIdx.x; idx < R * H; idx += 256) {
      const int r = idx / H, h = idx - r * H;
      as[idx] = load_as_f32(ap + r * fa.stride_r + h);
    }
    __syncthreads();
    // db: four neighbouring d per thread
    for (int idx = threadIdx.x; idx < (R << d4sh); idx += 256) {
      const int r = idx >> d4sh, d4 = idx & d4mask;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      for (int h = 0; h < H; ++h) {
        const f32x4 xv = *reinterpret_cast<const f32x4*>(xs + h * XS + 4 * d4);
        const float av = as[r * H + h];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += xv[e] * av;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) store_from_f32(ob + r * gb.stride_r + 4 * d4 + e, acc[e] * inv);
    }
    // da: ns = 1 << nsh neighbouring lanes share an output
    const int per_pass = 256 >> nsh, sub = threadIdx.x & ((1 << nsh) - 1);
    for (int base = 0; base < R * H; base += per_pass) {  // uniform trip count: the shuffles below need every lane
      const int idx = base + (threadIdx.x >> nsh);
      const bool ok = idx < R * H;
      const int r = ok ? idx / H : 0, h = ok ? idx - r * H : 0;
      float acc = 0.f;
      for (int d = 4 * sub; d < D; d += 4 << nsh) {
        const f32x4 xv = *reinterpret_cast<const f32x4*>(xs + h * XS + d);
        const f32x4 bv = *reinterpret_cast<const f32x4*>(bs + r * D + d);
        acc += xv[0] * bv[0] + xv[1] * bv[1] + xv[2] * bv[2] + xv[3] * bv[3];
      }
      for (int m = (1 << nsh) >> 1; m >= 1; m >>= 1) acc += __shfl_xor(acc, m, 64);
      if (ok && sub == 0) store_from_f32(oa + r * ga.stride_r + h, acc * inv);
    }
  } else {
    for (int idx = threadIdx.x; idx < R * D; idx += 256) {
      const int r = idx / D, d = idx - r * D;
      float acc = 0.f;
      for (int h = 0; h < H; ++h) acc += xp[h * D + d] * load_as_f32(ap + r * fa.stride_r + h);
      store_from_f32(ob + r * gb.stride_r + d, acc * inv);
    }
    for (int idx = threadIdx.x; idx < R * H; idx += 256) {
      const int r = idx / H, h = idx - r * H;
      float acc = 0.f;
      for (int d = 0; d < D; ++d) acc += xp[h * D + d] * load_as_f32(bp + r * fb.stride_r + d);
      store_from_f32(oa + r * ga.stride_r + h, acc * inv);
    }
  }
}

// The same projections for factors with H % 8 == 0 and (D / 8) (H / 8) a power of two up to 64,
// without LDS: a thread owns an 8 x 8 piece of one token's dX, rows 8 hg .. 8 hg + 7, columns 4 cc .. 4 cc + 3 of
// the lower and of the upper half of D (pieces of D are the fastest thread index, so each of the 16 loads of a
// piece reads whole contiguous half rows across the lanes: 12 % faster than 8 consecutive columns per thread,
// where one load instruction touched every other 16 bytes), multiplies it
// with its 8 values of b (for da) and of a (for db) rank by rank, and the sums over d and over h are
// reductions across the lanes that share a token: over the D / 8 neighbouring lanes with DPP adds,
// over the H / 8 groups above them with DPP adds and exchanges of rows of lanes, in registers throughout: through the LDS
// (ds_bpermute, eight or more per rank) the kernel waited for them, 1340 tokens x 16 heads x 128 with ranks 6, 2, 2 took 14.7 us
// instead of 11.1 us, 16 384 x 32 x 64 93 instead of 79 (403 MB read, 5 TB/s: at that size the memory is what bounds it).
// Several tokens share a wave.
// All arrays that this kernel takes in one launch (blockIdx.z): at short lengths a launch of its own leaves each of them
// waiting for the one before.  The gradients are written in the type the caller wants them in (rounded once, from the fp32 sums).
struct ProjectJob { const float* dx; TpaFactor fa, fb; TpaGrad ga, gb; int L, R, D; };
struct ProjectJobs { ProjectJob job[3]; int first[3], ranks, blocks, B; };  // array i: blockIdx.z = first[i] on, `ranks` ranks for each; blocks > 0: batch entries of so many workgroups, one after the other in blockIdx.x
template <typename T>
using Four = std::conditional_t<sizeof(T) == 2, u32x2, f32x4>;  // four values as they lie in memory
__device__ __forceinline__ f32x4 as_f32(const u32x2& x) { return f32x4{bf16lo_to_f32(x[0]), bf16hi_to_f32(x[0]), bf16lo_to_f32(x[1]), bf16hi_to_f32(x[1])}; }
__device__ __forceinline__ f32x4 as_f32(const f32x4& x) { return x; }
template <typename TO>
__device__ __forceinline__ void store_four(TO* p, f32x4 x) {
  if constexpr (sizeof(TO) == 2) *reinterpret_cast<u32x2*>(p) = u32x2{pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3])};
  else *reinterpret_cast<f32x4*>(p) = x;
}
template <typename TO>
__device__ __forceinline__ void store_two(TO* p, float x, float y) {
  if constexpr (sizeof(TO) == 2) *reinterpret_cast<uint32_t*>(p) = pack_bf16(x, y);
  else p[0] = x, p[1] = y;
}
template <typename TO>
__device__ __forceinline__ void store_eight(TO* p, const float* x) {
  if constexpr (sizeof(TO) == 2) {
    *reinterpret_cast<u32x4*>(p) = u32x4{pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]), pack_bf16(x[4], x[5]), pack_bf16(x[6], x[7])};
  } else {
    *reinterpret_cast<f32x4*>(p) = f32x4{x[0], x[1], x[2], x[3]};
    *reinterpret_cast<f32x4*>(p + 4) = f32x4{x[4], x[5], x[6], x[7]};
  }
}
// x and y of the lanes N apart: the lanes of the lower side get the sum of the two x, those of the upper side that of the two y
template <int N>
__device__ __forceinline__ float swap_add(float x, float y) {
  const unsigned a = __float_as_uint(x), b = __float_as_uint(y);
  auto s = N == 16 ? __builtin_amdgcn_permlane16_swap(a, b, false, false) : __builtin_amdgcn_permlane32_swap(a, b, false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
template <typename T, typename TO>
__global__ __launch_bounds__(256) void project_h8_kernel(ProjectJobs jobs, int H) {
  const int z = blockIdx.z, job = (z >= jobs.first[1]) + (z >= jobs.first[2]);
  const ProjectJob j = job == 0 ? jobs.job[0] : job == 1 ? jobs.job[1] : jobs.job[2];
  const int r0 = (z - (job == 0 ? jobs.first[0] : job == 1 ? jobs.first[1] : jobs.first[2])) * jobs.ranks;
  const TpaFactor &fa = j.fa, &fb = j.fb;
  const TpaGrad &ga = j.ga, &gb = j.gb;
  const int L = j.L, R = j.R, D = j.D;
  const int cpr = D / 8, hgs = H / 8, tt = cpr * hgs;  // threads per token
  int cc, hg;
  int64_t tok;
  int blk = blockIdx.x, b = blockIdx.y;
  if (jobs.blocks > 0) {
    b = blk / jobs.blocks;
    blk -= b * jobs.blocks;
    if (b >= jobs.B) return;
  }
  piece_of(cpr, hgs, tok, hg, cc, blk);
  const bool live = tok < L;
  if ((int64_t)blk * (256 >> __builtin_ctz(tt)) >= L) return;  // a whole workgroup past the end of a shorter array
  const int64_t t = live ? tok : L - 1;  // lanes past the end idle along: the reductions need whole waves
  const int dh = D / 2;  // a thread's eight columns: 4 cc .. 4 cc + 3 and the same in the upper half of the row
  const float* xp = j.dx + (((int64_t)b * L + t) * H + 8 * hg) * D + 4 * cc;
  const T* ap = static_cast<const T*>(fa.ptr) + b * fa.stride_b + t * fa.stride_l + 8 * hg;
  const T* bp = static_cast<const T*>(fb.ptr) + b * fb.stride_b + t * fb.stride_l + 4 * cc;
  float x[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const f32x4 lo = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(xp + (int64_t)i * D));
    const f32x4 hi = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(xp + (int64_t)i * D + dh));
#pragma unroll
    for (int j = 0; j < 4; ++j) { x[i][j] = lo[j]; x[i][4 + j] = hi[j]; }
  }
  const float inv = 1.f / (float)R;
  // which of the lanes that share a (token, piece of D) write which of its columns, see db below
  const int swaps = (tt > 16) + (tt > 32), lane = threadIdx.x & 63;
  const bool writes = live && (cpr == 16 || (lane & 8) == 0);
  const int column = (lane & 16 ? dh : 0) + (swaps == 2 && (lane & 32) ? 2 : 0);
  TO* oa = reinterpret_cast<TO*>(ga.ptr) + b * ga.stride_b + t * ga.stride_l + 8 * hg;
  TO* ob = reinterpret_cast<TO*>(gb.ptr) + b * gb.stride_b + t * gb.stride_l + 4 * cc;
  // a rank's factors are requested while the one before is worked on (two ranks ahead: the small sizes gain 0.3 us, but the
  // registers cost a wave per SIMD and 16 384 tokens x 32 heads x 64 go from 81 to 84 us)
  Four<T> next[4];
  auto request = [&](int r) __attribute__((always_inline)) {
    const T* const a = ap + (int64_t)r * fa.stride_r;
    const T* const b = bp + (int64_t)r * fb.stride_r;
    next[0] = *reinterpret_cast<const Four<T>*>(a);
    next[1] = *reinterpret_cast<const Four<T>*>(a + 4);
    next[2] = *reinterpret_cast<const Four<T>*>(b);
    next[3] = *reinterpret_cast<const Four<T>*>(b + dh);
  };
  request(r0);
  const int r1 = min(R, r0 + jobs.ranks);
  for (int r = r0; r < r1; ++r) {
    const f32x4 al = as_f32(next[0]), ah = as_f32(next[1]), bl = as_f32(next[2]), bh = as_f32(next[3]);
    if (r + 1 < r1) request(r + 1);
    float af[8], bf[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) { af[j] = al[j]; af[4 + j] = ah[j]; bf[j] = bl[j]; bf[4 + j] = bh[j]; }
    float da[8], db[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc += x[i][j] * bf[j];
      da[i] = acc;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc += x[i][j] * af[i];
      db[j] = acc;
    }
    // da: sum over the cpr (8 or 16) neighbouring lanes of this (token, head group)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float v = da[i];
      v = dpp_add<0xB1>(v);   // quad_perm [1, 0, 3, 2]
      v = dpp_add<0x4E>(v);   // quad_perm [2, 3, 0, 1]
      v = dpp_add<0x141>(v);  // row_half_mirror: the other quad of the same eight lanes
      if (cpr == 16) v = dpp_add<0x140>(v);  // row_mirror: the other eight lanes of the row
      da[i] = v * inv;
    }
    if (live && cc == 0) store_eight(oa + (int64_t)r * ga.stride_r, da);
    // db: sum over the head groups, which lie cpr lanes apart.  The exchange of two rows of 16 lanes (or of the two halves of
    // the wave) takes a pair of values and leaves each side the sum of one of them, so that the lanes share out the columns
    if (cpr == 8 && hgs > 1) {
#pragma unroll
      for (int j = 0; j < 8; ++j) db[j] = dpp_add<0x128>(db[j]);  // row_ror 8: the other eight lanes of the row
    }
    TO* const o = ob + (int64_t)r * gb.stride_r;
    if (swaps == 0) {
      if (live && hg == 0) {
        store_four(o, f32x4{db[0] * inv, db[1] * inv, db[2] * inv, db[3] * inv});
        store_four(o + dh, f32x4{db[4] * inv, db[5] * inv, db[6] * inv, db[7] * inv});
      }
      continue;
    }
    float h4[4];  // odd rows of the wave: columns of the upper half
#pragma unroll
    for (int j = 0; j < 4; ++j) h4[j] = swap_add<16>(db[j], db[j + 4]);
    if (swaps == 1) {
      if (writes) store_four(o + column, f32x4{h4[0] * inv, h4[1] * inv, h4[2] * inv, h4[3] * inv});
      continue;
    }
    const float lo = swap_add<32>(h4[0], h4[2]), hi = swap_add<32>(h4[1], h4[3]);  // upper half of the wave: columns 2, 3 of the four
    if (writes) store_two(o + column, lo * inv, hi * inv);
  }
}

inline bool al16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }
// rows of whole 16-byte pieces
template <typename T>
bool rows16(const TpaFactor& f) {
  constexpr int N = 16 / sizeof(T);
  return al16(f.ptr) && f.stride_b % N == 0 && f.stride_l % N == 0 && f.stride_r % N == 0;
}

// Whether project_h8_kernel takes an array: each is judged by itself, so that one that it cannot take (an unaligned view,
// another head size) does not send the others to the kernel of one workgroup per token.
template <typename T, typename TO>
bool projects_by_h8(const ProjectJob& j, int H) {
  const int cpr = j.D / 8, tt = cpr * (H / 8);
  const TpaFactor ga{j.ga.ptr, j.ga.stride_b, j.ga.stride_l, j.ga.stride_r}, gb{j.gb.ptr, j.gb.stride_b, j.gb.stride_l, j.gb.stride_r};
  return j.D % 8 == 0 && H % 8 == 0 && (cpr == 8 || cpr == 16) && tt <= 64 && (tt & (tt - 1)) == 0 && ((int64_t)j.L * tt + 255) / 256 <= 2147483647LL &&
         al16(j.dx) && rows16<T>(j.fa) && rows16<T>(j.fb) && rows16<TO>(ga) && rows16<TO>(gb);
}

// Ranks that a workgroup of the launch takes.  One after the other they are a chain of 0.6 us each that a short call has too few workgroups
// to hide, so there they are dealt to workgroups of their own, which read dx again, as long as these are no more than 400.  us, all ranks / so,
// by workgroups of one array: ranks 16, 8, 8: 11 of them (335 tokens, 8 heads of 64) 14.9 / 6.5, 63 17.1 / 12.5 (four ranks each, 504 workgroups
// 11.7), 99 19.0 / 15.8 (four each 19.0), 250 23.4 / 25.8; 6, 2, 2: 34 7.2 / 5.3, 54 7.8 / 7.2, fp32 64 8.6 / 7.0; 6, 4, 4: 175 13.1 / 13.5.
// That holds where the parts of a token find its dx in the L2 of their XCD: workgroups go to the XCDs in turn, so a part has a multiple of eight of them (the
// last ones past every array), those of all batch entries side by side.  Without that, whole backward, all ranks / parts of two: ranks 6, 4, 4, 3 x 156 tokens, 32 heads of 64 (60 workgroups)
// 29.9 / 34.2, 2 x 218 (56) 30.4 / 28.1; 4, 3, 3, 208 tokens, 64 heads (52) 26.8 / 32.3, 2 x 112 (56) 27.0 / 26.0; 6, 2, 2, 3 x 130, 64 heads (99) 31.5 /
// 32.3, 16 x 164, 8 heads (96) 29.6 / 27.4.
int ranks_per_workgroup(const ProjectJobs& jobs, unsigned n, int64_t blocks) {
  int most = 0;
  for (unsigned i = 0; i < n; ++i) most = std::max(most, jobs.job[i].R);
  for (int k = std::min(most / 2, 16); k > 1; --k) {
    const int ranks = (most + k - 1) / k;
    int64_t parts = 0;
    for (unsigned i = 0; i < n; ++i) parts += (jobs.job[i].R + ranks - 1) / ranks;
    if (blocks * parts <= 400) return ranks;
  }
  return most;
}

template <typename T, typename TO>
void launch_project(const ProjectJobs& jobs, int B, int H, hipStream_t stream) {
  ProjectJobs h8{};
  int64_t blocks = 0;
  unsigned n = 0;
  for (const ProjectJob& j : jobs.job) {
    if (projects_by_h8<T, TO>(j, H)) {
      h8.job[n++] = j;
      blocks = std::max(blocks, ((int64_t)j.L * (j.D / 8) * (H / 8) + 255) / 256);
      continue;
    }
    const size_t smem = ((size_t)H * (j.D + 4) + (size_t)j.R * j.D + (size_t)j.R * H) * sizeof(float);
    int dsh = 0;
    while ((1 << dsh) < j.D) ++dsh;
    int nsh = 0;  // lanes per da output: a power of two, at most a wave, so that one pass covers the outputs if it can
    while (nsh < 6 && (4 << nsh) * j.R * H <= 512 && (16 << nsh) <= j.D) ++nsh;
    if (smem <= 60 * 1024 && (1 << dsh) == j.D && j.D >= 4)
      hipLaunchKernelGGL((project_kernel<T, TO, true>), dim3(j.L, B), dim3(256), smem, stream, j.dx, j.fa, j.fb, j.ga, j.gb, j.L, H, j.D, j.R, dsh, nsh);
    else
      hipLaunchKernelGGL((project_kernel<T, TO, false>), dim3(j.L, B), dim3(256), 0, stream, j.dx, j.fa, j.fb, j.ga, j.gb, j.L, H, j.D, j.R, dsh, nsh);
  }
  if (!n) return;
  h8.ranks = ranks_per_workgroup(h8, n, blocks * B);
  unsigned parts = 0;
  for (unsigned i = 0; i < 3; ++i) {
    h8.first[i] = i < n ? (int)parts : INT32_MAX;
    if (i < n) parts += (h8.job[i].R + h8.ranks - 1) / h8.ranks;
  }
  dim3 grid((unsigned)blocks, B, parts);
  if (parts > n) {
    h8.blocks = (int)blocks;
    h8.B = B;
    grid = dim3((unsigned)((blocks * B + 7) / 8 * 8), 1, parts);
  }
  hipLaunchKernelGGL((project_h8_kernel<T, TO>), grid, dim3(256), 0, stream, h8, H);
}

template <typename T, int DMAX>
int launch_dense_t(const DenseParams& p, hipStream_t stream) {
  constexpr int kTile = tile_of(DMAX);
  const size_t smem_q = (size_t)kTile * (p.dk + p.dv) * sizeof(float) + kTile * sizeof(int);
  const size_t smem_kv = (size_t)kTile * (p.dk + p.dv + 2) * sizeof(float) + kTile * sizeof(int);
  hipLaunchKernelGGL((bwd_dq_kernel<T, DMAX>), dim3((p.lq + kThreads - 1) / kThreads, p.H, p.B), dim3(kThreads), smem_q, stream, p);
  if (hipGetLastError() != hipSuccess) return TPA_ERR_LAUNCH;
  hipLaunchKernelGGL((bwd_dkv_kernel<T, DMAX>), dim3((p.lk + kThreads - 1) / kThreads, p.H, p.B), dim3(kThreads), smem_kv, stream, p);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

template <typename T>
int launch_dense(const DenseParams& p, hipStream_t stream) {
  const int dmax = p.dk > p.dv ? p.dk : p.dv;
  if (dmax <= 8) return launch_dense_t<T, 8>(p, stream);
  if (dmax <= 32) return launch_dense_t<T, 32>(p, stream);
  if (dmax <= 64) return launch_dense_t<T, 64>(p, stream);
  if (dmax <= 128) return launch_dense_t<T, 128>(p, stream);
  if (dmax <= 256) return launch_dense_t<T, 256>(p, stream);
  return TPA_ERR_SHAPE;
}

inline size_t align256(size_t n) { return (n + 255) & ~size_t(255); }

template <typename T>
int tpa_bwd_t(const TpaBwdArgs* a, hipStream_t stream, bool mfma) {
  const size_t nq = (size_t)a->B * a->lq * a->H * a->dk, nk = (size_t)a->B * a->lk * a->H * a->dk,
               nv = (size_t)a->B * a->lk * a->H * a->dv, nd = (size_t)a->B * a->H * a->lq;
  char* w = static_cast<char*>(a->workspace);
  auto take = [&](size_t floats) { float* ptr = reinterpret_cast<float*>(w); w += align256(floats * sizeof(float)); return ptr; };
  // dense Q, K, V (fp32, or bf16 for the MFMA kernels: then only half of each slot is used)
  float *qd = take(nq), *kd = take(nk), *vd = take(nv), *dqd = take(nq), *dkd = take(nk), *dvd = take(nv), *delta = take(nd);

  const int threads = 256;
  // the matrix-core kernels: bf16 ones on bf16 copies of Q, K, V; fp32 ones on the fp32 copies
  const bool mfma32 = mfma && sizeof(T) == sizeof(float);
  mfma = mfma && !mfma32;
  // dense Q, K, V and delta in one launch where the vectorised kernels apply (16-byte aligned arrays, H % 8 == 0, a row
  // of D on 8, 16 or 32 lanes)
  const int cpr = a->dk * (int)sizeof(T) / 16;
  bool one_launch = (mfma || mfma32) && a->H % 8 == 0 && a->dk == a->dv && cpr >= 8 && cpr <= 32 && (cpr & (cpr - 1)) == 0 &&
                    a->dk * sizeof(T) % 16 == 0 && al16(a->o) && al16(a->d_o);
  const TpaFactor* fs[6] = {&a->qa, &a->qb, &a->ka, &a->kb, &a->va, &a->vb};
  for (const TpaFactor* f : fs) one_launch = one_launch && rows16<T>(*f);
  const int lmax = a->lq > a->lk ? a->lq : a->lk;
  const int64_t blocks = ((int64_t)lmax * cpr * (a->H / 8) + 255) / 256;
  int32_t *qwin = nullptr, *kwin = nullptr;
  if (one_launch && blocks <= 2147483647LL) {
    ReconJobs jobs{};
    jobs.job[0] = ReconJob{a->qa, a->qb, qd, a->lq, a->rq, 1.f, a->lq, nullptr};
    jobs.job[1] = ReconJob{a->ka, a->kb, kd, a->lk, a->rk, 1.f, a->lk, nullptr};
    jobs.job[2] = ReconJob{a->va, a->vb, vd, a->lk, a->rk, 1.f, a->lk, nullptr};
    jobs.delta = DeltaJob{a->o, a->d_o, delta, a->lq};
    if (mfma && a->q_segment_ids && windows_ahead_pay(a->B, a->H, a->lq, a->lk, a->rk >= 16 ? 512 : 8192)) {
      // into the halves of the slots of Q and K that bf16 leaves: H D / 2 words a row there, eight a block taken
      const int block = dense_bwd_mfma_block(a->B, a->lq, a->lk, a->H, a->dk, a->causal, 1), coff = causal_offset_of(a);
      qwin = reinterpret_cast<int32_t*>(qd + nq / 2);
      kwin = reinterpret_cast<int32_t*>(kd + nk / 2);
      jobs.windows[0] = WindowJob{a->q_segment_ids, a->kv_segment_ids, nullptr, a->lq, a->lk, block, 0, a->causal != 0, coff, qwin, (a->lq + block - 1) / block * 8, 8, 0, 1};
      jobs.windows[1] = WindowJob{a->kv_segment_ids, a->q_segment_ids, nullptr, a->lk, a->lq, block, 1, a->causal != 0, coff, kwin, (a->lk + block - 1) / block * 8, 8, 0, 1};
    }
    if constexpr (sizeof(T) == 2) hipLaunchKernelGGL(recon_bf16_h8_kernel, dim3((unsigned)blocks, a->B, 4), dim3(256), 0, stream, jobs, a->H, a->dk);
    else hipLaunchKernelGGL(recon_f32_h8_kernel, dim3((unsigned)blocks, a->B, 4), dim3(256), 0, stream, jobs, a->H, a->dk);
  } else {
    if (mfma) {
      auto recon16 = [&](const TpaFactor& fa, const TpaFactor& fb, float* slot, int L, int D, int R) {
        uint16_t* out = reinterpret_cast<uint16_t*>(slot);
        if (sizeof(T) == 2 && rows16<uint16_t>(fb))
          hipLaunchKernelGGL(recon_bf16_kernel, dim3((L + kReconTokens - 1) / kReconTokens, a->B), dim3(threads), 0, stream, fa, fb, out, L, a->H, D, R, 1.f);
        else
          hipLaunchKernelGGL((recon_kernel<T, uint16_t>), dim3(L, a->B), dim3(threads), 0, stream, fa, fb, out, L, a->H, D, R);
      };
      recon16(a->qa, a->qb, qd, a->lq, a->dk, a->rq);
      recon16(a->ka, a->kb, kd, a->lk, a->dk, a->rk);
      recon16(a->va, a->vb, vd, a->lk, a->dv, a->rk);
    } else {
      hipLaunchKernelGGL((recon_kernel<T, float>), dim3(a->lq, a->B), dim3(threads), 0, stream, a->qa, a->qb, qd, a->lq, a->H, a->dk, a->rq);
      hipLaunchKernelGGL((recon_kernel<T, float>), dim3(a->lk, a->B), dim3(threads), 0, stream, a->ka, a->kb, kd, a->lk, a->H, a->dk, a->rk);
      hipLaunchKernelGGL((recon_kernel<T, float>), dim3(a->lk, a->B), dim3(threads), 0, stream, a->va, a->vb, vd, a->lk, a->H, a->dv, a->rk);
    }
    const int vec = a->dv % 8 == 0 && al16(a->o) && al16(a->d_o);
    hipLaunchKernelGGL((delta_kernel<T>), dim3((unsigned)((nd * 16 + threads - 1) / threads)), dim3(threads), 0, stream,
                       static_cast<const T*>(a->o), static_cast<const T*>(a->d_o), delta, a->B, a->lq, a->H, a->dv, vec);
  }
  if (hipGetLastError() != hipSuccess) return TPA_ERR_LAUNCH;

  int rc;
  if (mfma) {
    rc = dense_bwd_mfma_launch(qd, kd, vd, a->d_o, a->lse, delta, a->q_segment_ids, a->kv_segment_ids, dqd, dkd, dvd,
                               a->B, a->lq, a->lk, a->H, a->dk, a->sm_scale, a->causal, causal_offset_of(a), qwin, kwin, stream);
  } else if (mfma32) {
    rc = dense_bwd_f32_launch(qd, kd, vd, static_cast<const float*>(a->d_o), a->lse, delta, a->q_segment_ids, a->kv_segment_ids,
                              dqd, dkd, dvd, a->B, a->lq, a->lk, a->H, a->dk, a->sm_scale, a->causal, causal_offset_of(a), stream);
  } else {
    DenseParams p{};
    p.q = qd; p.k = kd; p.v = vd; p.d_o = a->d_o; p.lse = a->lse; p.delta = delta;
    p.qseg = a->q_segment_ids; p.kvseg = a->kv_segment_ids; p.bias = nullptr;
    p.dq = dqd; p.dk_out = dkd; p.dv_out = dvd;
    p.B = a->B; p.lq = a->lq; p.lk = a->lk; p.H = a->H; p.dk = a->dk; p.dv = a->dv;
    p.sm_scale = a->sm_scale; p.causal = a->causal; p.coff = causal_offset_of(a);
    rc = launch_dense<T>(p, stream);
  }
  if (rc != TPA_OK) return rc;

  const ProjectJobs jobs{{{dqd, a->qa, a->qb, a->dqa, a->dqb, a->lq, a->rq, a->dk},
                          {dkd, a->ka, a->kb, a->dka, a->dkb, a->lk, a->rk, a->dk},
                          {dvd, a->va, a->vb, a->dva, a->dvb, a->lk, a->rk, a->dv}}};
  if (sizeof(T) == 2 && a->grad_dtype == TPA_DTYPE_BF16) {
    if constexpr (sizeof(T) == 2) launch_project<T, uint16_t>(jobs, a->B, a->H, stream);
  } else {
    launch_project<T, float>(jobs, a->B, a->H, stream);
  }
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

template <typename T>
int mha_bwd_t(const MhaBwdArgs* a, hipStream_t stream, bool mfma) {
  const size_t nq = (size_t)a->B * a->lq * a->H * a->dk, nk = (size_t)a->B * a->lk * a->H * a->dk,
               nv = (size_t)a->B * a->lk * a->H * a->dv, nd = (size_t)a->B * a->H * a->lq;
  char* w = static_cast<char*>(a->workspace);
  auto take = [&](size_t floats) { float* ptr = reinterpret_cast<float*>(w); w += align256(floats * sizeof(float)); return ptr; };
  float* delta = take(nd);
  const int threads = 256;
  {
    const int vec = a->dv % 8 == 0 && !(reinterpret_cast<uintptr_t>(a->o) & 15) && !(reinterpret_cast<uintptr_t>(a->d_o) & 15);
    hipLaunchKernelGGL((delta_kernel<T>), dim3((unsigned)((nd * 16 + threads - 1) / threads)), dim3(threads), 0, stream,
                       static_cast<const T*>(a->o), static_cast<const T*>(a->d_o), delta, a->B, a->lq, a->H, a->dv, vec);
  }
  if (hipGetLastError() != hipSuccess) return TPA_ERR_LAUNCH;
  if (mfma && sizeof(T) == sizeof(float))
    return dense_bwd_f32_launch(static_cast<const float*>(a->q), static_cast<const float*>(a->k), static_cast<const float*>(a->v),
                                static_cast<const float*>(a->d_o), a->lse, delta, nullptr, nullptr, a->dq, a->dk_out, a->dv_out,
                                a->B, a->lq, a->lk, a->H, a->dk, a->sm_scale, a->causal, 0, stream);
  if (mfma)
    return dense_bwd_mfma_launch(a->q, a->k, a->v, a->d_o, a->lse, delta, nullptr, nullptr, a->dq, a->dk_out, a->dv_out,
                                 a->B, a->lq, a->lk, a->H, a->dk, a->sm_scale, a->causal, 0, nullptr, nullptr, stream);
  const float *qd, *kd, *vd;
  if constexpr (sizeof(T) == sizeof(float)) {
    qd = static_cast<const float*>(a->q); kd = static_cast<const float*>(a->k); vd = static_cast<const float*>(a->v);
  } else {
    float *q32 = take(nq), *k32 = take(nk), *v32 = take(nv);
    auto blocks = [&](size_t n) { return dim3((unsigned)((n + threads - 1) / threads < 65535 * 16 ? (n + threads - 1) / threads : 65535 * 16)); };
    hipLaunchKernelGGL((to_f32_kernel<T>), blocks(nq), dim3(threads), 0, stream, static_cast<const T*>(a->q), q32, (int64_t)nq);
    hipLaunchKernelGGL((to_f32_kernel<T>), blocks(nk), dim3(threads), 0, stream, static_cast<const T*>(a->k), k32, (int64_t)nk);
    hipLaunchKernelGGL((to_f32_kernel<T>), blocks(nv), dim3(threads), 0, stream, static_cast<const T*>(a->v), v32, (int64_t)nv);
    qd = q32; kd = k32; vd = v32;
  }
  if (hipGetLastError() != hipSuccess) return TPA_ERR_LAUNCH;
  DenseParams p{};
  p.q = qd; p.k = kd; p.v = vd; p.d_o = a->d_o; p.lse = a->lse; p.delta = delta;
  p.qseg = nullptr; p.kvseg = nullptr; p.bias = a->bias;
  p.dq = a->dq; p.dk_out = a->dk_out; p.dv_out = a->dv_out;
  p.B = a->B; p.lq = a->lq; p.lk = a->lk; p.H = a->H; p.dk = a->dk; p.dv = a->dv;
  p.sm_scale = a->sm_scale; p.causal = a->causal;
  return launch_dense<T>(p, stream);
}

}  // namespace
}  // namespace tpa

int tpa_recon_dense_bf16(const TpaFactor* fa, const TpaFactor* fb, uint16_t* out, int B, int L, int H, int D, int R, float scale, hipStream_t stream) {
  if (B > 65535) return TPA_ERR_SHAPE;
  const bool vec = D % 8 == 0 && !(reinterpret_cast<uintptr_t>(fb->ptr) & 15) && fb->stride_b % 8 == 0 && fb->stride_l % 8 == 0 &&
                   fb->stride_r % 8 == 0;
  const bool vec_a = vec && H % 8 == 0 && !(reinterpret_cast<uintptr_t>(fa->ptr) & 15) && fa->stride_b % 8 == 0 && fa->stride_l % 8 == 0 &&
                     fa->stride_r % 8 == 0;
  const int64_t threads = (int64_t)L * (D / 8) * (H / 8);
  if (vec_a && (threads + 255) / 256 <= 2147483647LL) {
    tpa::ReconJobs jobs{};
    jobs.job[0] = tpa::ReconJob{*fa, *fb, out, L, R, scale, L, nullptr};
    hipLaunchKernelGGL(tpa::recon_bf16_h8_kernel, dim3((unsigned)((threads + 255) / 256), B, 1), dim3(256), 0, stream, jobs, H, D);
  } else if (vec)
    hipLaunchKernelGGL(tpa::recon_bf16_kernel, dim3((L + tpa::kReconTokens - 1) / tpa::kReconTokens, B), dim3(256), 0, stream, *fa, *fb, out, L, H, D, R, scale);
  else if (scale != 1.f)
    return TPA_ERR_ALIGN;  // the scaled form exists for 16-byte aligned factors only
  else
    hipLaunchKernelGGL((tpa::recon_kernel<uint16_t, uint16_t>), dim3(L, B), dim3(256), 0, stream, *fa, *fb, out, L, H, D, R);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

// Q (with its scale), K and V in one launch where every factor is 16-byte aligned and H % 8 == 0;
// TPA_ERR_UNSUPPORTED otherwise (the caller then reconstructs them one by one).
bool tpa_recon_dense_qkv_takes(const TpaFwdArgs* a) {
  if (a->B > 65535 || a->H % 8 != 0 || a->dk % 8 != 0 || a->dk != a->dv) return false;
  const TpaFactor* fs[6] = {&a->qa, &a->qb, &a->ka, &a->kb, &a->va, &a->vb};
  for (const TpaFactor* f : fs)
    if ((reinterpret_cast<uintptr_t>(f->ptr) & 15) || f->stride_b % 8 != 0 || f->stride_l % 8 != 0 || f->stride_r % 8 != 0) return false;
  return true;
}

int tpa_recon_dense_qkv_bf16(const TpaFwdArgs* a, uint16_t* qd, uint16_t* kd, uint16_t* vd, float q_scale, const tpa::WindowJob& windows, hipStream_t stream) {
  if (!tpa_recon_dense_qkv_takes(a)) return TPA_ERR_UNSUPPORTED;
  const int lmax = a->lq > a->lk ? a->lq : a->lk;
  const int64_t blocks = ((int64_t)lmax * (a->dk / 8) * (a->H / 8) + 255) / 256;
  if (blocks > 2147483647LL) return TPA_ERR_UNSUPPORTED;
  const int keys = tpa::keys_in_reach(a);
  tpa::ReconJobs jobs{};
  jobs.job[0] = tpa::ReconJob{a->qa, a->qb, qd, a->lq, a->rq, q_scale, a->lq, nullptr};
  jobs.job[1] = tpa::ReconJob{a->ka, a->kb, kd, a->lk, a->rk, 1.f, keys, a->kv_lengths};
  jobs.job[2] = tpa::ReconJob{a->va, a->vb, vd, a->lk, a->rk, 1.f, keys, a->kv_lengths};
  jobs.windows[0] = windows;
  hipLaunchKernelGGL(tpa::recon_bf16_h8_kernel, dim3((unsigned)blocks, a->B, 3), dim3(256), 0, stream, jobs, a->H, a->dk);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

namespace {
int64_t recon_f32_blocks(const TpaFwdArgs* a) { return ((int64_t)(a->lq > a->lk ? a->lq : a->lk) * (a->dk / 4) * (a->H / 8) + 255) / 256; }
}  // namespace

bool tpa_recon_dense_qkv_f32_takes(const TpaFwdArgs* a) {
  if (a->B > 65535 || a->H % 8 != 0 || a->dk != a->dv || (a->dk != 64 && a->dk != 128) || recon_f32_blocks(a) > 2147483647LL) return false;
  const TpaFactor* fs[6] = {&a->qa, &a->qb, &a->ka, &a->kb, &a->va, &a->vb};
  for (const TpaFactor* f : fs)
    if (!tpa::rows16<float>(*f)) return false;
  return true;
}

int tpa_recon_dense_qkv_f32(const TpaFwdArgs* a, float* qd, float* kd, float* vd, float q_scale, hipStream_t stream) {
  if (!tpa_recon_dense_qkv_f32_takes(a)) return TPA_ERR_UNSUPPORTED;
  const int64_t blocks = recon_f32_blocks(a);
  const int keys = tpa::keys_in_reach(a);
  tpa::ReconJobs jobs{};
  jobs.job[0] = tpa::ReconJob{a->qa, a->qb, qd, a->lq, a->rq, q_scale, a->lq, nullptr};
  jobs.job[1] = tpa::ReconJob{a->ka, a->kb, kd, a->lk, a->rk, 1.f, keys, a->kv_lengths};
  jobs.job[2] = tpa::ReconJob{a->va, a->vb, vd, a->lk, a->rk, 1.f, keys, a->kv_lengths};
  hipLaunchKernelGGL(tpa::recon_f32_h8_kernel, dim3((unsigned)blocks, a->B, 3), dim3(256), 0, stream, jobs, a->H, a->dk);
  return hipGetLastError() == hipSuccess ? TPA_OK : TPA_ERR_LAUNCH;
}

size_t tpa_bwd_workspace_size(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t dk, int64_t dv) {
  using tpa::align256;
  const size_t nq = (size_t)(B * lq * H * dk), nk = (size_t)(B * lk * H * dk), nv = (size_t)(B * lk * H * dv), nd = (size_t)(B * H * lq);
  return 2 * (align256(nq * 4) + align256(nk * 4) + align256(nv * 4)) + align256(nd * 4);
}

size_t mha_bwd_workspace_size(int64_t B, int64_t lq, int64_t lk, int64_t H, int64_t dk, int64_t dv, int dtype) {
  using tpa::align256;
  const size_t nq = (size_t)(B * lq * H * dk), nk = (size_t)(B * lk * H * dk), nv = (size_t)(B * lk * H * dv), nd = (size_t)(B * H * lq);
  size_t bytes = align256(nd * 4);
  if (dtype != TPA_DTYPE_F32) bytes += align256(nq * 4) + align256(nk * 4) + align256(nv * 4);
  return bytes;
}

int tpa_bwd_launch(const TpaBwdArgs* a, hipStream_t stream, int mfma) {
  if (a->B > 65535 || a->H > 65535) return TPA_ERR_SHAPE;
  if (a->dtype == TPA_DTYPE_F32) return tpa::tpa_bwd_t<float>(a, stream, mfma != 0);
  if (a->dtype == TPA_DTYPE_BF16) return tpa::tpa_bwd_t<uint16_t>(a, stream, mfma != 0);
  return TPA_ERR_DTYPE;
}

int mha_bwd_launch(const MhaBwdArgs* a, hipStream_t stream, int mfma) {
  if (a->B > 65535 || a->H > 65535) return TPA_ERR_SHAPE;
  if (a->dtype == TPA_DTYPE_F32) return tpa::mha_bwd_t<float>(a, stream, mfma != 0);
  if (a->dtype == TPA_DTYPE_BF16) return tpa::mha_bwd_t<uint16_t>(a, stream, mfma != 0);
  return TPA_ERR_DTYPE;
}
