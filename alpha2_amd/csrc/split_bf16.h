// fp32 products on the bf16 matrix pipes, shared by gemm_f32.hip and attention.hip.
//
// An fp32 value x is cut into three bf16 numbers h = bf16(x), m = bf16(x - h), l = bf16(x - h - m), each rounded to nearest:
// 8 + 8 + 8 bits hold the 24 of an fp32 significand, so h + m + l IS x.  A product x y is accumulated in fp32 as
//     l h' + h l' + m m' + m h' + h m' + h h'
// (what is left out, m l' + l m' + l l', is at most 2^-24 |x y| and of either sign): six v_mfma_f32_32x32x16_bf16 of 32 cycles
// for 16 steps of the contraction where eight v_mfma_f32_32x32x2_f32 take 512.  The method is that of G. Henry, P. T. P. Tang
// and A. Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype for Higher-Precision Computations", ARITH 2019.
//
// Both operands are multiplied by 2^24 before the cut and the sums by 2^-48 after it: every fp32 number is a multiple of 2^-149,
// so every part is a multiple of 2^-125 and none is subnormal, which bf16 holds in fewer bits (unscaled, the parts of a number of
// 2^-112 are 1e-7 of it off, of 2^-120 2.5e-5 and of 2^-126 1.6e-3).  Where a value times 2^24 rounds to infinity (from 2^104 on), or a short sum
// times 2^48 does (from 2^80 on), or an operand is infinite or NaN, the sum is not finite: a workgroup that finds one computes its
// results again with the fp32 instruction, and those stand.
#pragma once
#include "common.h"

namespace ah {

constexpr float SPLIT_UP = 0x1p24f, SPLIT_DOWN = 0x1p-48f;

// A value that was loaded under a condition (zero past the end of a row), where it is used: the compiler would multiply it in the branch
// that loads it otherwise, and wait for it there.
__device__ __forceinline__ float here(float x) {
  asm("" : "+v"(x));
  return x;
}
struct Split2 { uint32_t h, m, l; };       // the parts of two values side by side
// x less the low (high) half of h: v_dot2_f32_bf16 with (-1, 0) or (0, -1), in place of an instruction that makes an fp32 number of the
// half and one that subtracts it: nine instructions for a pair of values in place of 13 (2.0 ns of a SIMD each where a shift takes 1.9 and
// a subtraction 1.2).  The result is exact for every significand (times 1, each comes out of a product as it went in: all of them, at
// eight pairs of exponents of the two halves), and the other half, unless it is infinite or NaN, adds nothing.  The constants are hidden from the compiler, which takes 0xbf80 in the
// low half alone for the one in both.
__device__ __forceinline__ uint32_t hidden(uint32_t c) {
  asm("" : "+s"(c));
  return c;
}
__device__ __forceinline__ float less_low(float x, uint32_t h) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, h), __builtin_bit_cast(bf16x2_t, hidden(0x0000bf80u)), x, false);
}
__device__ __forceinline__ float less_high(float x, uint32_t h) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, h), __builtin_bit_cast(bf16x2_t, hidden(0xbf800000u)), x, false);
}
// x0, x1: values that are already multiplied by SPLIT_UP
__device__ __forceinline__ Split2 split2(float x0, float x1) {
  Split2 s;
  s.h = pack_bf16x2(x0, x1);
  x0 = less_low(x0, s.h);
  x1 = less_high(x1, s.h);
  s.m = pack_bf16x2(x0, x1);
  x0 = less_low(x0, s.m);
  x1 = less_high(x1, s.m);
  s.l = pack_bf16x2(x0, x1);
  return s;
}
// 8 consecutive values of a contraction (times SPLIT_UP) as operands
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8 (&f)[3]) {
  uint32_t w[3][4];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const Split2 s = split2(x[2 * e], x[2 * e + 1]);
    w[0][e] = s.h; w[1][e] = s.m; w[2][e] = s.l;
  }
#pragma unroll
  for (int p = 0; p < 3; p++) f[p] = __builtin_bit_cast(bf16x8, make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]));
}
// the parts that are multiplied, first and second operand, the smallest product first
constexpr int SPLIT_A[6] = {2, 0, 1, 1, 0, 0}, SPLIT_B[6] = {0, 2, 1, 0, 1, 0};
// acc += the six products; element (row of a, column of b)
__device__ __forceinline__ void mfma6(const bf16x8 (&a)[3], const bf16x8 (&b)[3], f32x16 &acc) {
#pragma unroll
  for (int p = 0; p < 6; p++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[SPLIT_A[p]], b[SPLIT_B[p]], acc, 0, 0, 0);
}
__device__ __forceinline__ bool all_finite(const f32x16 &acc) {
  float z = 0.f;
#pragma unroll
  for (int e = 0; e < 16; e++) z = __builtin_fmaf(acc[e], 0.f, z);      // 0 unless one is infinite or NaN
  return z == 0.f;
}
template <int N>
__device__ __forceinline__ bool all_finite(const f32x16 (&acc)[N]) {
  bool fine = true;
#pragma unroll
  for (int d = 0; d < N; d++) fine = fine && all_finite(acc[d]);
  return fine;
}

}  // namespace ah
