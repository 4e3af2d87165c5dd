// fp32 products on the bf16 matrix cores: an fp32 number as the exact sum of
// three bf16 numbers, and the product of two such sums.
#pragma once

#include "tv_common.h"

namespace tv {

// x = h + m + l in bf16: h and m are x and x - h rounded to eight bits, and what
// is then left fits a third, so the sum is exact.  (Henry, Tang and Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019, describe such splits.)  Rounding to nearest gives m
// and l a sign of their own: with parts that are cut off, every left-out product
// has the sign of the whole one and a sum of them grows with its length.  An
// infinite or NaN x leaves NaN parts, which the caller's result shows.
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  auto bits = [](float x) { return __builtin_bit_cast(uint32_t, x); };
  h = pack2<__bf16>(a, b);
  a -= bf16_lo(h);
  b -= bf16_hi(h);
  m = pack2<__bf16>(a, b);
  l = __builtin_amdgcn_perm(bits(b - bf16_hi(m)), bits(a - bf16_lo(m)), 0x07060302u);   // upper halves: the rest is zero
}

// Operands are scaled by 2^24 before they are split: the lowest bit of the
// smallest fp32 number (2^-149) is then a normal bf16 number, so the sum of the
// parts is exact for every operand and not only above 2^-110, whatever the
// matrix core does with subnormals.  Operands of 2^104 and more overflow, and so
// do sums of 2^80 and more; the caller sees both as results that are not finite
// and repeats them in plain fp32.
constexpr float kSplitScale = 0x1p24f;
constexpr float kSplitUnscale = 0x1p-48f;   // of a product of two

// Split eight operands.
__device__ __forceinline__ void split8(f32x4 a, f32x4 b, u32x4 (&s)[3]) {
  a *= kSplitScale;
  b *= kSplitScale;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint32_t h, m, l;
    split2(a[2 * i], a[2 * i + 1], h, m, l);
    s[0][i] = h; s[1][i] = m; s[2][i] = l;
    split2(b[2 * i], b[2 * i + 1], h, m, l);
    s[0][2 + i] = h; s[1][2 + i] = m; s[2][2 + i] = l;
  }
}
__device__ __forceinline__ f32x4 as_f32x4(u32x4 w) { return __builtin_bit_cast(f32x4, w); }

// c += 2^48 A B from the parts of both, smallest products first.  The three products
// of the lowest parts are left out: at most 0.992 * 2^-24 of the whole product
// (the largest over all 2^23 significands, m = 1 - 2^-8 half steps), zero on
// average.
constexpr int kSplitProducts = 6;
constexpr int kSplitA[kSplitProducts] = {2, 0, 1, 1, 0, 0};
constexpr int kSplitB[kSplitProducts] = {0, 2, 1, 0, 1, 0};
__device__ __forceinline__ f32x4 mfma_split(const u32x4 (&a)[3], const u32x4 (&b)[3], f32x4 c) {
#pragma unroll
  for (int q = 0; q < kSplitProducts; ++q) c = mfma16x16x32<__bf16>(a[kSplitA[q]], b[kSplitB[q]], c);
  return c;
}

}  // namespace tv
