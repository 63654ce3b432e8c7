// fp32 products on the bf16 matrix cores: every fp32 operand is written as
// the sum of three bf16 pieces (8 significand bits each, 24 together), and a
// product a b is accumulated in fp32 from six of the nine piece products (the
// method of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial
// intelligence datatype for higher-precision computations", ARITH 2019).
//
//   a = a0 + a1 + a2,  a0 = bf16(a), a1 = bf16(a - a0), a2 = a - a0 - a1
//   a b ~ a0 b2 + a2 b0 + a1 b1 + a0 b1 + a1 b0 + a0 b0
//
// The pieces are round-to-nearest, so |a1| <= 2^-8 |a| and |a2| <= 2^-17 |a|:
// the split is exact (no operand bit is dropped) and the three products left
// out are at most 2^-24 |a b| together, one fp32 rounding (0.99 of it at a = b =
// 0x1.00ff8p+0); their root mean square over the significands is 2^-27.5 |a b|.
// So a product that stands alone has a largest error of 2 x 2^-24, measured
// 1.77 (fp32 MFMA 1.00), and the same root mean square, 0.42.
// gfx950's 32x32x16 bf16 MFMA runs 16 times the rate of the 32x32x2 fp32 one,
// so six of them take 6/16 of the time, and it rounds its accumulator once
// per 16 products where the fp32 one rounds once per 2.  Measured against
// float64 on one 32x32 tile of N(0,1) operands with one accumulator (relative
// 2-norm error, fp32 MFMA -> this): K = 16 7.4e-8 -> 3.4e-8, 64 1.5e-7 ->
// 1.1e-7, 512 4.1e-7 -> 3.4e-7, 4096 1.2e-6 -> 1.0e-6, 16384 2.3e-6 -> 2.1e-6;
// uniform [0, 1) operands 6.2e-8 -> 3.2e-8, ..., 1.7e-6 -> 1.1e-6.
//
// Operands are scaled by kSplitUp = 2^24 before they are split, and the sums by
// kSplitDown = 2^-48 (all exact): the last piece then stays above bf16's
// smallest subnormal, 2^-133, for every fp32 operand down to 2^-134, so a
// gradient's or a softmax's tails keep their bits.  bf16 MFMA keeps subnormal
// operands.  What the split cannot hold is flagged and computed by fp32 MFMA
// instead: infinities, NaN and operands past 2^103 (their remainder is NaN),
// operands below 2^-134 (their remainder is an fp32 subnormal), and sums past
// 2^80, which overflow.
#pragma once
#include "common.h"

namespace nship {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

// Two floats rounded to nearest bf16, packed (x low): one v_cvt_pk_bf16_f32
// (converted element by element, x is converted twice).
__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{x, y}, bf16x2));
}
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

constexpr float kSplitUp = 0x1p24f, kSplitDown = 0x1p-48f;

// signaling / quiet NaN, -inf, +inf, -subnormal, +subnormal
constexpr int kUnsplittable = 0x1 | 0x2 | 0x4 | 0x200 | 0x10 | 0x80;

// The three pieces of a pair, each packed (a low).
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& p0, uint32_t& p1, uint32_t& p2) {
  p0 = pack_bf16(a, b);
  const float ra = a - bf16_lo(p0), rb = b - bf16_hi(p0);
  p1 = pack_bf16(ra, rb);
  p2 = pack_bf16(ra - bf16_lo(p1), rb - bf16_hi(p1));
}
// ... and `bad` set when either value cannot be split (see above).
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& p0, uint32_t& p1, uint32_t& p2, bool& bad) {
  p0 = pack_bf16(a, b);
  const float ra = a - bf16_lo(p0), rb = b - bf16_hi(p0);
  p1 = pack_bf16(ra, rb);
  const float sa = ra - bf16_lo(p1), sb = rb - bf16_hi(p1);
  bad |= __builtin_amdgcn_classf(sa, kUnsplittable) | __builtin_amdgcn_classf(sb, kUnsplittable);
  p2 = pack_bf16(sa, sb);
}

// W floats (a multiple of 4) -> W / 2 packed words of each piece.
template <int W>
__device__ __forceinline__ void split_run(const float* v, uint32_t (&p0)[W / 2], uint32_t (&p1)[W / 2],
                                          uint32_t (&p2)[W / 2], bool& bad) {
#pragma unroll
  for (int j = 0; j < W / 2; j++) split_pair(v[2 * j], v[2 * j + 1], p0[j], p1[j], p2[j], bad);
}

// The six piece products of step q: A piece kPieceA[q] with B piece
// kPieceB[q], smallest first.
constexpr int kPieceA[6] = {0, 2, 1, 0, 1, 0};
constexpr int kPieceB[6] = {2, 0, 1, 1, 0, 0};

}  // namespace nship
