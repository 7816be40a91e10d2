// f32 products on the bf16 matrix cores (the method of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", 2019). A float is the exact sum of three bf16 parts (8 + 8 + 8
// significand bits):
// h = bf16(x), m = bf16(x - h), l = x - h - m, all rounded to nearest, so |m| <= 2^-8 |x| and |l| <= 2^-16 |x|. The
// product of two such sums is nine bf16 products; the six of order up to 2^-16 are kept,
//   x y = l h' + h l' + m m' + m h' + h m' + h h',
// each exact in the f32 accumulator, and the dropped three (m l', l m', l l') are about 2^-23 |x y| at most (their
// bounds add up to (1 + 2^-9) 2^-23), 2^-26 on average and of either sign. Six 32x32x16 bf16 MFMAs take 192 cycles for 16 k where eight 32x32x2 f32 MFMAs take 512, and
// they round the accumulator six times per 16 k instead of eight: against float64, 32 x 32 dot products of N(0, 1)
// values are off by 1.6e-7 / 4.3e-7 / 9.5e-7 (2-norm) at K = 128 / 768 / 3072, on f32 MFMAs by 2.1e-7 / 4.9e-7 / 1.0e-6.
//
// A bf16 part keeps bits down to 2^-133, so the operands that kernels split themselves and the GEMM's stored weights are
// multiplied by 2^23 first (exact, and the sum by its inverse at the end): every float down to the smallest denormal is then
// the exact sum of its parts. Winograd's stored U is not scaled (its parts sum to U). An element that three parts cannot
// hold, 2^105 and above of a scaled operand or below 2^-110 of an unscaled one, is stored as a NaN part with its bits behind
// it, and its columns are recomputed in f32: 2 to 4.8 times the GEMM's time where that took every tile, which is why the
// weights are scaled: small ones do occur.
//
// An infinite or NaN element, or one that times 2^23 rounds past the largest bf16, splits into parts of which one is NaN,
// and so makes every output it enters NaN; two finite elements whose product f32 still holds may have h h' past it (both
// round up, or by the scale), which leaves an infinity. Kernels test their sums for either and recompute such tiles on f32
// MFMAs, which gives the value the f32 sum has.
#pragma once

#include <hip/hip_runtime.h>

namespace lkd {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 0x1p23f;     // of the parts that split3 makes
constexpr float kSplitUnscale = 0x1p-23f;  // of a sum with one such operand; squared with two

// the parts of scale a and scale b (scale kSplitScale, or 0 for elements past the operand's end) as bf16 pairs (a in the
// low half)
__device__ __forceinline__ void split3(float a, float b, float scale, unsigned& h, unsigned& m, unsigned& l) {
  a *= scale;
  b *= scale;
  h = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a, b}), bf16x2));
  const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{ra, rb}), bf16x2));
  l = __builtin_bit_cast(unsigned, __builtin_convertvector(
                                       (f32x2{ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u)}),
                                       bf16x2));
}

__device__ __forceinline__ void split3(f32x4 x, float scale, u32x2& h, u32x2& m, u32x2& l) {
  unsigned a[3], b[3];
  split3(x[0], x[1], scale, a[0], a[1], a[2]);
  split3(x[2], x[3], scale, b[0], b[1], b[2]);
  h = u32x2{a[0], b[0]};
  m = u32x2{a[1], b[1]};
  l = u32x2{a[2], b[2]};
}

// An operand fragment of a 32x32x16 MFMA (8 consecutive k of one row or column per lane) in its three parts.
struct Frag3 {
  bf16x8 h, m, l;
};

__device__ __forceinline__ Frag3 split3(f32x4 x0, f32x4 x1, float scale) {
  u32x2 h0, m0, l0, h1, m1, l1;
  split3(x0, scale, h0, m0, l0);
  split3(x1, scale, h1, m1, l1);
  return Frag3{__builtin_bit_cast(bf16x8, (u32x4{h0[0], h0[1], h1[0], h1[1]})),
               __builtin_bit_cast(bf16x8, (u32x4{m0[0], m0[1], m1[0], m1[1]})),
               __builtin_bit_cast(bf16x8, (u32x4{l0[0], l0[1], l1[0], l1[1]}))};
}

// acc += a b over 16 k, the smallest products first
__device__ __forceinline__ f32x16 mfma3(const Frag3& a, const Frag3& b, f32x16 acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.l, b.h, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.l, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.m, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.h, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.m, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.h, acc, 0, 0, 0);
}

// The same in two accumulators, the h h' products in hi and the five smaller ones, about 2^-7 of it at most, in lo: hi is rounded
// once per 16 k instead of six times (a third of the error at the same speed, for 16 more registers).
__device__ __forceinline__ void mfma3(const Frag3& a, const Frag3& b, f32x16& hi, f32x16& lo) {
  lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.l, b.h, lo, 0, 0, 0);
  lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.l, lo, 0, 0, 0);
  hi = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.h, hi, 0, 0, 0);
  lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.m, lo, 0, 0, 0);
  lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.h, lo, 0, 0, 0);
  lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.m, lo, 0, 0, 0);
}

// The three bf16 parts of 8 values as splitExact stores them, in r[0 .. 2], become the values themselves, in r[0] and r[1];
// unscale the inverse of its scale.
__device__ __forceinline__ void joinParts(f32x4 (&r)[3], float unscale) {
  const u32x4 h = __builtin_bit_cast(u32x4, r[0]), m = __builtin_bit_cast(u32x4, r[1]);
  const u32x4 l = __builtin_bit_cast(u32x4, r[2]);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      const auto high = [&](unsigned x) { return o ? x & 0xffff0000u : x << 16; };
      const auto f = [&](unsigned x) { return __uint_as_float(high(x)); };
      const unsigned bits = high(m[i]) | high(l[i]) >> 16;
      r[i >> 1][2 * (i & 1) + o] =
          f(h[i]) != f(h[i]) && bits ? __uint_as_float(bits) : ((f(h[i]) + f(m[i])) + f(l[i])) * unscale;
    }
}

// The parts of scale v (scale 1 or kSplitScale) for 8 values of an operand that is stored split, for every float: parts of
// a value that would round past the largest bf16 are cut instead of rounded, infinities and NaN are h alone, and a value
// that the scale takes past the largest float, or with bits below 2^-133, is h = NaN with the float's own two halves in m
// and l, so that joinParts gives it back.
__device__ __forceinline__ void splitExact(const float (&v)[8], float scale, u32x4 (&parts)[3]) {
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    constexpr float kMax = 3.40282347e38f;
    float rest = v[k] * scale;
    const bool finite = fabsf(rest) <= kMax, cut = fabsf(rest) >= 3.38953139e38f;
    unsigned part[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const unsigned b = __float_as_uint(rest);
      part[q] = (cut || !finite ? b : b + 0x7fff + ((b >> 16) & 1)) >> 16;
      rest = finite ? rest - __uint_as_float(part[q] << 16) : 0.0f;
    }
    if (v[k] != v[k]) part[0] |= 0x40;  // a NaN whose bits are all in the low half
    if (rest != 0.0f || (!finite && fabsf(v[k]) <= kMax)) {
      const unsigned b = __float_as_uint(v[k]);
      part[0] = 0x7fc0;
      part[1] = b >> 16;
      part[2] = b & 0xffff;
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) parts[q][k >> 1] = k & 1 ? parts[q][k >> 1] | part[q] << 16 : part[q];
  }
}

}  // namespace lkd
