// The dropout mask of ah_dropout_mask, element by element: shared by elementwise.hip and the LayerNorms of nn.hip.
#pragma once
#include "common.h"

namespace ah {

// DropoutRng.hash of the reference's CPU path (packages/autograd/src/ops.ts:74-81), bit for bit: the first line is evaluated in
// doubles, one rounding per operation (no fused multiply-add), and only then cut to 32 bits, so products past 2^53 have already
// lost low bits exactly as a JS number does.  (The reference's own GPU kernel wraps in u32 instead,
// packages/helios/src/kernels/nn.ts:5600-5748, and so differs from its CPU path for element indices above ~4.0 M.)
// The sum is an integer-valued double below 2^63: the int64 conversion is exact and its low 32 bits are ToInt32.
// For indices below `whole` neither product nor sum passes 2^53, so the doubles are exact and the low 32 bits are those of whole-number
// arithmetic: one addition an element and one multiplication for four, where the conversions, product, sum and remainder in doubles took about
// a dozen instructions and bound the kernel, not memory.  h 2^-32 > p is h > p 2^32, a comparison of whole numbers with its floor.  Applying a mask
// to 3.9 M bf16 elements 6.5 -> 4.9 us, with a residual 7.9 -> 6.9; past `whole` (4.0 M for small counters) as before with the comparison gained.
struct DropMask { uint32_t whole, above; float keep; };
inline DropMask drop_mask(int32_t counter, double p) {
  const double left = 9007199254740992.0 - 2147483648.0 - (counter < 0 ? -(double)counter : (double)counter) * 2654435761.0;
  return {left > 0 ? (uint32_t)(left / 2246822519.0) : 0u, (uint32_t)(p * 4294967296.0), (float)(1.0 / (1.0 - p))};
}
struct DropBase { double sum; uint32_t low; };
__device__ __forceinline__ DropBase drop_base(int32_t seed, int32_t counter) {
#pragma clang fp contract(off)
  return {(double)seed + (double)counter * 2654435761.0, (uint32_t)seed + (uint32_t)counter * 2654435761u};
}
__device__ __forceinline__ float drop_factor(uint32_t h, const DropMask &m) {
  h = (h ^ (h >> 16)) * 0x85ebca6bu;
  h = (h ^ (h >> 13)) * 0xc2b2ae35u;
  h = h ^ (h >> 16);
  return h > m.above ? m.keep : 0.f;
}
// the factors of elements i .. i + N - 1
template <int N>
__device__ __forceinline__ void drop_keep(const DropBase &base, uint32_t i, const DropMask &m, float (&keep)[N]) {
#pragma clang fp contract(off)
  if (i < m.whole && N - 1 < m.whole - i) {
    const uint32_t low = base.low + i * 2246822519u;
#pragma unroll
    for (int e = 0; e < N; e++) keep[e] = drop_factor(low + e * 2246822519u, m);
  } else {
#pragma unroll
    for (int e = 0; e < N; e++) keep[e] = drop_factor((uint32_t)(int64_t)(base.sum + (double)(i + e) * 2246822519.0), m);
  }
}

}  // namespace ah
