// fp32 contractions on the bf16 matrix cores.
//
// A float is the exact sum of three bf16 numbers, x = h + m + l (8 + 8 + 8 bits, each the rounding of what the ones before
// it leave), so a product of two floats is the sum of nine products of bf16 numbers, all exact in fp32.  Six of them are
// formed, h h, h m, m h, m m, h l and l h; the three dropped ones are below 2^-24 of the product.  The sums are fp32, and a
// v_mfma_f32_32x32x16_bf16 adds sixteen products at a time where v_mfma_f32_32x32x2_f32 rounds after every two: against 64
// bits the split is the more accurate of the two (N(0, 1) operands, relative rms error of dot products of length 64 / 128 /
// 1024: fp32 units 1.4e-7 / 2.0e-7 / 5.7e-7, in two chains 1.1e-7 / 1.5e-7 / 4.1e-7; split 1.1e-7 / 1.6e-7 / 4.9e-7, with the
// five small terms in an accumulator of their own 0.5e-7 / 0.65e-7 / 1.9e-7).  Six steps of 32 cycles do the work of eight of
// 64.
//
// (The split and the choice of six products: G. Henry, P. T. P. Tang and A. Heinecke, Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations, arXiv 1904.06376.)
//
// The split needs its parts to be numbers of bf16's range.  The matrix cores keep denormals, in operands, products and sums, so at
// the small end it is exact down to 2^-110, where the last bit of a value is the spacing of bf16's denormals.  A workgroup that
// meets an infinity, a NaN, a value that rounds up to infinity or one nonzero value below 2^-90 (2^20 away from that, for the
// weights that are made from the products of such values) walks all its tiles a second time with the fp32 instruction on whole
// floats; `Magnitudes` tells.  That costs what the fp32 instruction costs and the first walk on top: forward and backward of 2 x 1000
// tokens, 8 heads of 64, causal 131 us, 211 where every workgroup of the backward walks twice, 170 with the fp32 instruction alone; 8 x
// 2000, 16 heads 1.9, 4.7 and 3.1 ms.  The weights themselves (p, dS) are split wherever they lie: those below 2^-110 have an absolute
// error of at most 2^-134.
#pragma once

#include "tpa_common.h"

namespace tpa {

typedef __attribute__((ext_vector_type(4))) uint32_t split_words;
struct Split3 { bf16x8 h, m, l; };  // one MFMA operand
struct Pair3 { uint32_t h, m, l; };  // two floats

// a - (float)(one half of `pair`): the other half is multiplied by zero
__device__ __forceinline__ Pair3 split_pair(float a, float b) {
  // -1 in the low / in the high half; kept from the assembler's inline constants, which name the high half of a pair
  uint32_t lo = 0x0000bf80u, hi = 0xbf800000u;
  asm("" : "+s"(lo), "+s"(hi));
  auto less = [](uint32_t pair, uint32_t half, float x) __attribute__((always_inline)) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, half), x, false);
  };
  Pair3 r;
  r.h = pack_bf16(a, b);
  a = less(r.h, lo, a);
  b = less(r.h, hi, b);
  r.m = pack_bf16(a, b);
  r.l = pack_bf16(less(r.m, lo, a), less(r.m, hi, b));
  return r;
}

// Two floats whole, for the walk with the fp32 instruction: the upper and the lower halves of their bits
__device__ __forceinline__ Pair3 halves_of_pair(float a, float b) {
  const uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
  return {__builtin_amdgcn_perm(y, x, 0x07060302), __builtin_amdgcn_perm(y, x, 0x05040100), 0u};
}

template <bool FP32 = false>
__device__ __forceinline__ Split3 split8(const float (&x)[8]) {
  split_words h, m, l;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const Pair3 p = FP32 ? halves_of_pair(x[2 * j], x[2 * j + 1]) : split_pair(x[2 * j], x[2 * j + 1]);
    h[j] = p.h;
    m[j] = p.m;
    l[j] = p.l;
  }
  return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}
// a float from its halves
__device__ __forceinline__ float join(const Split3& x, int e) {
  const uint32_t h = __builtin_bit_cast(split_words, x.h)[e / 2], m = __builtin_bit_cast(split_words, x.m)[e / 2];
  return __uint_as_float(e & 1 ? __builtin_amdgcn_perm(h, m, 0x07060302) : __builtin_amdgcn_perm(h, m, 0x05040100));
}

// the larger of `so_far` and |a|, |b|; NaN if any of them is
__device__ __forceinline__ float largest(float so_far, float a, float b) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(so_far, fabsf(a)), fabsf(b));
}
__device__ __forceinline__ float largest(float so_far, const f32x4& x) { return largest(largest(so_far, x[0], x[1]), x[2], x[3]); }
__device__ __forceinline__ float smallest(float so_far, const f32x4& x) {
  auto less = [](float a, float b) __attribute__((always_inline)) { return __builtin_elementwise_minimum(a, fabsf(b)); };
  return less(less(less(less(so_far, x[0]), x[1]), x[2]), x[3]);
}
// Operands of the logits alone (Q and K of the forward): what a small one loses, 2^-134 of the other one, is below 2^-27 of a
// logit's unit while that is below this, whatever the small one is
constexpr float kLogitOperand = 0x1p100f;
// The largest and the smallest nonzero magnitude of what a thread has staged
struct Magnitudes {
  float top = 0.f;
  uint32_t low = ~0u;  // twice the bits (no sign), less one: zero comes out on top
  __device__ __forceinline__ void add(float a, float b) {
    top = largest(top, a, b);
    low = min(min(low, 2 * __float_as_uint(a) - 1), 2 * __float_as_uint(b) - 1);
  }
  __device__ __forceinline__ void add(const f32x4& x) {
    add(x[0], x[1]);
    add(x[2], x[3]);
  }
  __device__ __forceinline__ bool irregular() const { return !(top < 0x1p127f) || low < 2 * (uint32_t)((127 - 90) << 23) - 1; }
};
// of sums of products: one that left the range of floats on the way, of whose parts one may be -inf and another +inf
__device__ __forceinline__ bool too_large(const f32x16& x) {
  float top = 0.f;
#pragma unroll
  for (int v = 0; v < 16; v += 2) top = largest(top, x[v], x[v + 1]);
  return !(top < 0x1p127f);
}

__device__ __forceinline__ f32x16 mfma_bf16(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
// c_small takes the five small terms, c the large one (they may be the same)
__device__ __forceinline__ void mfma_small(const Split3& a, const Split3& b, f32x16& c) {
  c = mfma_bf16(a.l, b.h, c);
  c = mfma_bf16(a.h, b.l, c);
  c = mfma_bf16(a.m, b.m, c);
  c = mfma_bf16(a.m, b.h, c);
  c = mfma_bf16(a.h, b.m, c);
}
// the fp32 instruction on the same operands.  The barrier keeps the sums of an operand that lives across a loop from
// being formed ahead of it and held in registers for this rare path.
__device__ __forceinline__ void mfma_joined(Split3 a, Split3 b, f32x16& c) {
  asm volatile("" : "+v"(b.h), "+v"(b.m));
#pragma unroll
  for (int e = 0; e < 8; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(join(a, e), join(b, e), c, 0, 0, 0);
}

// A lane's value and the kernel's arguments for the second walk, which the compiler cannot tell to be those of the first: what
// both walks form from them would otherwise be held in registers from the one to the other.
__device__ __forceinline__ int again(int x) {
  asm volatile("" : "+v"(x));
  return x;
}
template <typename P>
__device__ __forceinline__ const __attribute__((address_space(4))) P* arguments_again() {
  const __attribute__((address_space(4))) P* args = (const __attribute__((address_space(4))) P*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  return args;
}

}  // namespace tpa
