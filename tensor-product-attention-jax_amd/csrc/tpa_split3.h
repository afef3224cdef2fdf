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
// The split needs its parts to be numbers of bf16's range.  Infinities and NaN, values that round up to infinity, and
// operands so small that the parts of a product would be denormal take the fp32 instruction instead, tile by tile:
// `irregular` tells them by the largest magnitude that a lane has staged.  `split_any` splits such values too, so that
// `join` gives them back (to 2^-133, the spacing of bf16's denormals).
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

// the same for any values: no part of one spoils the other, and an infinity has no lower parts
__device__ __forceinline__ Pair3 split_pair_any(float a, float b) {
  auto rest = [](float x, float part) __attribute__((always_inline)) { return fabsf(part) == INFINITY ? 0.f : x - part; };
  Pair3 r;
  r.h = pack_bf16(a, b);
  a = rest(a, bf16lo_to_f32(r.h));
  b = rest(b, bf16hi_to_f32(r.h));
  r.m = pack_bf16(a, b);
  r.l = pack_bf16(a - bf16lo_to_f32(r.m), b - bf16hi_to_f32(r.m));
  return r;
}

template <bool ANY = false>
__device__ __forceinline__ Split3 split8(const float (&x)[8]) {
  split_words h, m, l;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const Pair3 p = ANY ? split_pair_any(x[2 * j], x[2 * j + 1]) : split_pair(x[2 * j], x[2 * j + 1]);
    h[j] = p.h;
    m[j] = p.m;
    l[j] = p.l;
  }
  return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}
__device__ __forceinline__ float join(const Split3& x, int e) { return ((float)x.h[e] + (float)x.m[e]) + (float)x.l[e]; }

// the larger of `so_far` and |a|, |b|; NaN if any of them is
__device__ __forceinline__ float largest(float so_far, float a, float b) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(so_far, fabsf(a)), fabsf(b));
}
__device__ __forceinline__ bool irregular(float largest_magnitude) {
  return !(largest_magnitude < 0x1p127f) || (largest_magnitude < 0x1p-50f && largest_magnitude != 0.f);
}
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
  asm volatile("" : "+v"(b.h), "+v"(b.m), "+v"(b.l));
#pragma unroll
  for (int e = 0; e < 8; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(join(a, e), join(b, e), c, 0, 0, 0);
}

}  // namespace tpa
