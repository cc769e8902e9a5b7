// Fused causal flash attention, forward and backward, on the gfx950 matrix cores.
//
// Semantics (packages/helios/src/kernels/attention.ts:1-586; CPU chain packages/model/src/gpt.ts:255-279):
//   s = scale * q.k;  s = cap * tanh(s / cap) when cap > 0;  keys after the query are masked;
//   P = softmax(s);  O = P V;  LSE = max + log(sum exp).
//
// fp32 path: v_mfma_f32_32x32x2_f32; for head sizes up to 64 bf16 matrix instructions on three parts of every operand (below).
// One wave owns 32 query rows (forward, dQ) or 32 key rows (dK/dV), and the products are arranged so that the owned index is the accumulator COLUMN (= lane % 32):
//   forward / dQ : S^T[kv, q] = K Q^T, so a lane holds 16 kv entries of one query row and the running
//                  max / sum / rescale are per-lane scalars (one cross-half shuffle per tile);
//                  O^T[d, q] += V^T[d, kv] P^T[kv, q] takes P^T straight from the accumulator registers.
//   dK / dV      : S[q, kv] = Q K^T with the key as column; dV^T += dO^T P and dK^T += Q^T dS likewise.
// An accumulator element e of a 32x32 tile sits at row 8*(e/4) + 4*(lane/32) + e%4, column lane%32, and
// MFMA number (j, r) of a 32-deep contraction contracts rows {8j + r, 8j + 4 + r}: half lane/32 = h owns
// row 8j + 4h + r in the accumulator and must supply exactly that row as operand -> no data movement.
#include "attention_common.h"
#include "split_bf16.h"
#include <type_traits>

using namespace ah;

namespace {

constexpr int BC = 32;     // rows of the streamed tile per iteration
constexpr int WAVES = 4;   // 4 waves x 32 owned rows = 128 rows per block

// (finite for a cap whose inverse is past the range, so that a score of zero stays one)
__device__ __forceinline__ float inverse_cap(float cap) { return cap > 0.f ? fminf(1.0f / cap, 3.402823466e38f) : 0.f; }
__device__ __forceinline__ float softcap_fwd(float s, float cap, float inv_cap) { return cap > 0.f ? tanhf(s * inv_cap) * cap : s; }
__device__ __forceinline__ float softcap_both(float s, float cap, float inv_cap, float &slope) {
  const float t = cap > 0.f ? tanhf(s * inv_cap) : 0.f;
  slope = 1.0f - t * t;
  return cap > 0.f ? t * cap : s;
}

// cooperative load of a [32 x D] f32 tile (rows row0.., zero beyond `rows` and beyond feature hd) into LDS with pitch D+1
template <int D>
__device__ __forceinline__ void load_tile_f32(float *s, const float *__restrict__ base, int64_t st, int row0, int rows, float mul, int hd) {
  constexpr int P = D + 1, V4 = D / 4;
  for (int c = threadIdx.x; c < BC * V4; c += blockDim.x) {
    int r = c / V4, d4 = c % V4;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (row0 + r < rows && d4 * 4 < hd) x = *reinterpret_cast<const float4 *>(base + (int64_t)(row0 + r) * st + d4 * 4);
    float *p = s + r * P + d4 * 4;
    p[0] = x.x * mul; p[1] = x.y * mul; p[2] = x.z * mul; p[3] = x.w * mul;
  }
}

// ------------------------------------------------------------------------------------------ products on the bf16 matrix pipes
// The cut and the six products are those of the fp32 products (split_bf16.h).  Every accumulator that is a matrix instruction's
// takes at most 24 of them (one 64-feature score, or one tile of 32 rows) and is then added, rounded to nearest, to an fp32 one.
// The tile of 32 streamed rows is cut once for the four waves and laid out in LDS both ways, three planes each:
//   rows     [row][feature]                  an operand is 8 features of a row
//   columns  [feature][row'], row' = 16 j + 8 h + 4 i + r of row 16 j + 8 i + 4 h + r: an operand is the 8 rows whose scores the
//            lanes of half h hold in accumulator elements 8 j .. 8 j + 7, so that those go straight into the other operand
// 16-byte pieces are permuted within a row so that 16 lanes that read the same piece of 16 rows meet 64 different banks.
// A result that is not finite has the block computed again with the fp32 instruction, whose result stands; so does a score.
// 192 heads x 1024 x 64: dK and dV 945 -> 486 us, dQ 520 -> 316; 512 x 256 x 32: 112 -> 84 and 81 -> 60; 4 x 70 x 64: 29 -> 24 and
// 26 -> 20 (before both operands were scaled, which costs 1 % of the backward pass at 192 x 1024 x 64 and 3 to 6 % of smaller ones, and
// before the scores' functions ran side by side, below).
// Relative error against 64 bits at 4 x 512 x 64: dQ 4.6e-7 -> 3.7e-7, dK 6.4e-7 -> 3.8e-7, dV 6.0e-7 -> 3.3e-7.  What bounds it now is
// vector issue: tanh, exp and the cut of scores, K and V for every 32 x 32 tile beside 3072 cycles of matrix instructions.
template <int D>
struct SplitTile {                          // D = 32 or 64
  static constexpr int F = D / 32, PLANE = 64 * D, BYTES = 3 * PLANE;      // either layout
  // A thread's patch of the tile: rows 4 (t / 32) .. + 3, features F (t % 32) ..
  static __device__ __forceinline__ void load(float (&x)[4][F], const float *__restrict__ base, int64_t st, int row0, int rows, int hd) {
    const int g = threadIdx.x >> 5, f = F * (threadIdx.x & 31);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = row0 + 4 * g + r;
      const bool in = row < rows && f < hd;
      const float *p = base + (int64_t)row * st + f;
      if (F == 2) {
        const float2 v = in ? *reinterpret_cast<const float2 *>(p) : make_float2(0.f, 0.f);
        x[r][0] = v.x; x[r][F - 1] = v.y;
      } else {
        x[r][0] = in ? p[0] : 0.f;
      }
    }
  }
  // (ahead of the barrier in front of put: some of the cut then goes ahead of it too)
  static __device__ __forceinline__ void scale(float (&x)[4][F], float mul) {
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int d = 0; d < F; d++) x[r][d] = here(x[r][d]) * mul;
  }
  static __device__ __forceinline__ float largest(const float (&x)[4][F]) {
    float top = 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) top = F == 2 ? fmaxf(fmaxf(top, fabsf(x[r][0])), fabsf(x[r][F - 1])) : fmaxf(top, fabsf(x[r][0]));
    return top;
  }
  static __device__ __forceinline__ int row_ofs(int row, int chunk) { return row * 2 * D + ((chunk ^ ((row * D >> 7) & (D / 8 - 1))) << 4); }
  static __device__ __forceinline__ int col_ofs(int d, int chunk) { return d * 64 + ((chunk ^ ((d >> 2) & 3)) << 4); }
  static __device__ __forceinline__ uint32_t lows(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
  static __device__ __forceinline__ uint32_t highs(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
  // into the layouts that are asked for
  template <bool ROWS, bool COLS>
  static __device__ __forceinline__ void put(const float (&x)[4][F], char *rows, char *cols) {
    const int g = threadIdx.x >> 5, f = F * (threadIdx.x & 31);
    Split2 s[F][2];                         // rows (0, 1) and (2, 3) of a feature
#pragma unroll
    for (int d = 0; d < F; d++)
#pragma unroll
      for (int i = 0; i < 2; i++) s[d][i] = split2(x[2 * i][d], x[2 * i + 1][d]);
#pragma unroll
    for (int p = 0; p < 3; p++) {
      auto part = [&](int d, int i) { return p == 0 ? s[d][i].h : p == 1 ? s[d][i].m : s[d][i].l; };
      if (COLS) {
        const int chunk = 2 * (g >> 2) + (g & 1), half = 8 * ((g >> 1) & 1);
#pragma unroll
        for (int d = 0; d < F; d++) *reinterpret_cast<uint2 *>(cols + p * PLANE + col_ofs(f + d, chunk) + half) = make_uint2(part(d, 0), part(d, 1));
      }
      if (ROWS) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          char *q = rows + p * PLANE + row_ofs(4 * g + r, f >> 3) + (f & 7) * 2;
          const uint32_t a = part(0, r >> 1), b = part(F - 1, r >> 1);
          if (F == 2) *reinterpret_cast<uint32_t *>(q) = r & 1 ? highs(a, b) : lows(a, b);
          else *reinterpret_cast<uint16_t *>(q) = (uint16_t)(r & 1 ? a >> 16 : a);
        }
      }
    }
  }
  // 8 features 16 step + 8 half of row lane % 32; 8 rows (elements 8 j .. + 7 of the half) of feature d
  static __device__ __forceinline__ void get_row(const char *rows, int row, int chunk, bf16x8 (&f)[3]) {
#pragma unroll
    for (int p = 0; p < 3; p++) f[p] = *reinterpret_cast<const bf16x8 *>(rows + p * PLANE + row_ofs(row, chunk));
  }
  static __device__ __forceinline__ void get_col(const char *cols, int d, int chunk, bf16x8 (&f)[3]) {
#pragma unroll
    for (int p = 0; p < 3; p++) f[p] = *reinterpret_cast<const bf16x8 *>(cols + p * PLANE + col_ofs(d, chunk));
  }
  // a row of a wave's own, features 16 step + 8 half .. + 7; then times mul, and cut.  (All loads of a kernel's start come before the
  // first of these two: each waits for what it takes.)
  static __device__ __forceinline__ void row(const float *p, bool live, int hd, int lk, float (&x)[D / 16][8]) {
#pragma unroll
    for (int i = 0; i < D / 16; i++) {
      const int d = 16 * i + 8 * lk;
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
      if (live && d < hd) { a = *reinterpret_cast<const float4 *>(p + d); b = *reinterpret_cast<const float4 *>(p + d + 4); }
      x[i][0] = a.x; x[i][1] = a.y; x[i][2] = a.z; x[i][3] = a.w;
      x[i][4] = b.x; x[i][5] = b.y; x[i][6] = b.z; x[i][7] = b.w;
    }
  }
  static __device__ __forceinline__ void scale(float (&x)[D / 16][8], float mul) {
#pragma unroll
    for (int i = 0; i < D / 16; i++)
#pragma unroll
      for (int e = 0; e < 8; e++) x[i][e] = here(x[i][e]) * mul;
  }
  static __device__ __forceinline__ void cut(float (&x)[D / 16][8], float mul, bf16x8 (&f)[D / 16][3]) {
    scale(x, mul);
#pragma unroll
    for (int i = 0; i < D / 16; i++) split8(x[i], f[i]);
  }
  // acc[d][.] = alpha acc[d][.] + columns (features) x the weights in x (times SPLIT_UP)
  static __device__ __forceinline__ void contract_rows(const char *cols, const f32x16 &x, int lr, int lk, float alpha, f32x16 (&acc)[F]) {
    bf16x8 b[2][3];
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const float v[8] = {x[8 * j], x[8 * j + 1], x[8 * j + 2], x[8 * j + 3], x[8 * j + 4], x[8 * j + 5], x[8 * j + 6], x[8 * j + 7]};
      split8(v, b[j]);
    }
#pragma unroll
    for (int d = 0; d < F; d++) {
      f32x16 t;
#pragma unroll
      for (int e = 0; e < 16; e++) t[e] = 0.f;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        bf16x8 a[3];
        get_col(cols, 32 * d + lr, 2 * j + lk, a);
        mfma6(a, b[j], t);
      }
#pragma unroll
      for (int e = 0; e < 16; e++) acc[d][e] = __builtin_fmaf(acc[d][e], alpha, t[e]);
    }
  }
};
// The functions of a tile's 16 scores in straight-line code, all 16 at once: the library's tanh branches for every score, and so did the cap
// and the masks, so that the 16 ran one after the other.  Forward / backward (delta, dQ, dK and dV), us, before -> now: 512 heads x 256 x
// 32 51 / 168 -> 45 / 128, 192 x 1024 x 64 269 / 816 -> 240 / 697 (without a cap 239 / 763 -> 219 / 665; the scores all at a cap of 0.75
// 309 / 888 -> 262 / 736), 32 x 128 x 32 8.5 / 42 ->
// 7.3 / 34, 12 x 500 x 64 22 / 184 -> 20 / 140.  Results against 64 bits (4 x 256 x 32 and 4 x 512 x 64): the same without a cap, up to 46 %
// closer with one of 5 or 30; under a cap of 0.75 with nearly every score at it, dQ up to 12 % further off and down to 13 % closer.
// tanh in the form of Cephes' tanhf (Moshier): for |x| < TANH_SMALL x + x^3 P(x^2), P here the fifth-order polynomial of least relative error
// there (fitted by reweighted least squares, Lawson's method), beyond that 1 - 2 / (exp(2 |x|) + 1).  Last places off at most, over all
// values from 0.5 to 1: 0.73 and 1.63 (the library's tanhf 0.78 and 1.39; its two-part argument and a corrected exponential bring the
// second to 1.56 and cost 5 % of the forward pass where scores are large).
constexpr float TANH_SMALL = 0.625f, LOG2E = 1.44269502162933349609375f, LOG2E_REST = 1.925963033e-8f;
__device__ __forceinline__ float tanh_small(float x) {
  const float z = x * x;
  float p = -0.005704985465854406f;
  p = __builtin_fmaf(p, z, 0.02063908614218235f);
  p = __builtin_fmaf(p, z, -0.05373971536755562f);
  p = __builtin_fmaf(p, z, 0.13331441581249237f);
  p = __builtin_fmaf(p, z, -0.3333328068256378f);
  return __builtin_fmaf(x * z, p, x);
}
// 2^UP exp x, x not much above 0 and not below -1e9 (there, as for infinite x, NaN or infinity may come of it): the integer part of
// x log2 e, whose constant is held in two parts (Cody and Waite), goes into the exponent, 2 to the rest is the instruction's.  0.96 last
// places off at most, 0.306 root mean square (expf: 0.84, 0.300; a single exponential of x log2 e times what that rounds off: 1.25, 0.41).
template <int UP>
__device__ __forceinline__ float exp_of(float x) {
  const float n = __builtin_rintf(x * LOG2E), rest = __builtin_fmaf(x, LOG2E_REST, __builtin_fmaf(x, LOG2E, -n));
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(rest), (int)n + UP);
}
__device__ __forceinline__ float tanh_large(float x) {
  const float e = __builtin_amdgcn_exp2f(fabsf(x) * (2.0f * LOG2E));
  return copysignf(__builtin_fmaf(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f), x);
}
// Raw scores (times 2^48) scaled back by `factor` (split_cap_factor) and, with a cap, put through tanh: a score is cap times that
__device__ __forceinline__ void scores_tanh(f32x16 &s, float cap, float factor) {
#pragma clang fp contract(off)
#pragma unroll
  for (int e = 0; e < 16; e++) s[e] *= factor;
  if (!(cap > 0.f)) return;
  float top = 0.f;
#pragma unroll
  for (int e = 0; e < 16; e += 2) top = fmaxf(fmaxf(top, fabsf(s[e])), fabsf(s[e + 1]));
  if (__all(top < TANH_SMALL)) {                                   // (NaN: either way gives NaN)
#pragma unroll
    for (int e = 0; e < 16; e++) s[e] = tanh_small(s[e]);
  } else {
#pragma unroll
    for (int e = 0; e < 16; e++) { const float small = tanh_small(s[e]), large = tanh_large(s[e]); s[e] = fabsf(s[e]) < TANH_SMALL ? small : large; }
  }
}
__device__ __forceinline__ float split_cap_factor(float cap) { return (cap > 0.f ? inverse_cap(cap) : 1.0f) * SPLIT_DOWN; }
// (a cap whose factor is no normal number is left to the fp32 instruction)
__device__ __forceinline__ bool split_cap_ok(float cap) { return !(cap > 0x1p70f); }
// An infinite score has to be found before it is capped or weighed: what is made of it looks like any other.  (NaN shows in that.)  Either
// at the scores, or where the operands of all of them are below LARGE_OPERAND: 64 products of those, times 2^48, stay below 2^127.
__device__ __forceinline__ bool scores_finite(const f32x16 &s) {
  float top = 0.f;
#pragma unroll
  for (int e = 0; e < 16; e += 2) top = fmaxf(fmaxf(top, fabsf(s[e])), fabsf(s[e + 1]));
  return top < INFINITY;
}
constexpr float LARGE_OPERAND = 0x1p36f;
// quarter j of an accumulator of products, as it is stored
__device__ __forceinline__ float4 summed(const f32x16 &x, int j) {
  return make_float4(x[4 * j] * SPLIT_DOWN, x[4 * j + 1] * SPLIT_DOWN, x[4 * j + 2] * SPLIT_DOWN, x[4 * j + 3] * SPLIT_DOWN);
}

// ------------------------------------------------------------------------------------------ forward
// The 32 queries from q0 on of every wave that asks for them (`redo`, the same for a wave), keys below `end` (the same for the block)
template <int D>
__device__ void flash_fwd_exact(const FlashArgs &a, int bh, int q0, int end, bool redo, float *smem) {
  constexpr int P = D + 1, DB = D / 32;
  float *Ks = smem, *Vs = Ks + BC * P;
  int b = bh / a.H, h = bh % a.H;
  int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  int qi = q0 + lr;
  const float *Q = (const float *)a.q + b * a.q_sb + h * a.q_sh;
  const float *K = (const float *)a.k + b * a.k_sb + h * a.k_sh;
  const float *V = (const float *)a.v + b * a.v_sb + h * a.v_sh;
  const float inv_cap = inverse_cap(a.cap);

  float qreg[D / 2];                                  // Q[qi][2i + lk] * scale
#pragma unroll
  for (int i = 0; i < D / 2; i++) qreg[i] = qi < a.T && 2 * i + lk < a.hd ? Q[(int64_t)qi * a.q_st + 2 * i + lk] * a.scale : 0.f;

  f32x16 o[DB];
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int e = 0; e < 16; e++) o[d][e] = 0.f;
  float m = -INFINITY, l = 0.f;

  for (int kv0 = 0; kv0 < end; kv0 += BC) {
    __syncthreads();
    load_tile_f32<D>(Ks, K, a.k_st, kv0, a.T, 1.0f, a.hd);
    load_tile_f32<D>(Vs, V, a.v_st, kv0, a.T, 1.0f, a.hd);
    __syncthreads();
    if (!redo || kv0 > q0 + 31) continue;             // whole tile is in this wave's future (uniform per wave)
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; e++) s[e] = 0.f;
#pragma unroll
    for (int i = 0; i < D / 2; i++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(Ks[lr * P + 2 * i + lk], qreg[i], s, 0, 0, 0);
    float tmax = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      int kv = kv0 + 8 * (e >> 2) + 4 * lk + (e & 3);
      float x = softcap_fwd(s[e], a.cap, inv_cap);
      x = (kv > qi || kv >= a.T) ? -INFINITY : x;
      s[e] = x;
      tmax = fmaxf(tmax, x);
    }
    tmax = max_lane<32>(tmax);
    float m_new = fmaxf(m, tmax);
    float m_use = m_new == -INFINITY ? 0.f : m_new;   // rows with nothing visible yet stay at zero weight
    float alpha = expf(m - m_use);
    float psum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e++) { float p = expf(s[e] - m_use); s[e] = p; psum += p; }
    psum = add_lane<32>(psum);
    l = l * alpha + psum;
    m = m_new;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) o[d][e] *= alpha;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) {                  // MFMA (j = e/4, r = e%4): this half supplies kv row 8j + 4lk + r
        int kvr = 8 * (e >> 2) + 4 * lk + (e & 3);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(Vs[kvr * P + 32 * d + lr], s[e], o[d], 0, 0, 0);
      }
  }
  if (redo && qi < a.T) {
    float inv_l = l > 0.f ? 1.0f / l : 0.f;
    float *O = (float *)a.o + b * a.o_sb + h * a.o_sh + (int64_t)qi * a.o_st;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        float4 w = make_float4(o[d][4 * j] * inv_l, o[d][4 * j + 1] * inv_l, o[d][4 * j + 2] * inv_l, o[d][4 * j + 3] * inv_l);
        if (32 * d + 8 * j + 4 * lk < a.hd) *reinterpret_cast<float4 *>(O + 32 * d + 8 * j + 4 * lk) = w;
      }
    if (lk == 0) a.lse[((int64_t)b * a.H + h) * a.T + qi] = m + logf(l);
  }
}

// Two kernels compute the forward pass of head sizes up to 64, and a row's result does not depend on which: both do the operations
// below on the tiles of 32 keys in ascending order, each with the same operands and roundings.
// Raw scores of the tile at key kv0 (times 2^48, row = key, column = this lane's query qi) -> what scores_tanh makes of them, -infinity
// where masked; the column's largest score, which is cap_mul times that
__device__ __forceinline__ float cap_mul(const FlashArgs &a) { return a.cap > 0.f ? a.cap : 1.0f; }
__device__ __forceinline__ float tile_scores(f32x16 &s, const FlashArgs &a, float factor, int kv0, int qi, int lk) {
#pragma clang fp contract(off)
  scores_tanh(s, a.cap, factor);
  float top = -INFINITY;
  if (__all(kv0 + 31 <= qi && kv0 + 32 <= a.T)) {                  // nothing to mask
#pragma unroll
    for (int e = 0; e < 16; e++) top = fmaxf(top, s[e]);
  } else {
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int kv = kv0 + 8 * (e >> 2) + 4 * lk + (e & 3);
      s[e] = kv > qi || kv >= a.T ? -INFINITY : s[e];
      top = fmaxf(top, s[e]);
    }
  }
  return max_lane<32>(top) * cap_mul(a);
}
// Scores -> weights against the largest score so far, times 2^24; the column's sum of them, and what sums so far are multiplied by
// (-infinity, a masked score or no score so far, weighs what -200 does: nothing)
__device__ __forceinline__ float tile_weights(f32x16 &s, float mul, float before, float top, float &alpha) {
#pragma clang fp contract(off)
  const float m = fmaxf(before, top), use = m == -INFINITY ? 0.f : m;
  alpha = exp_of<0>(fmaxf(before - use, -200.f));
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 16; e++) { s[e] = exp_of<24>(fmaxf(__builtin_fmaf(s[e], mul, -use), -200.f)); sum += s[e]; }
  return add_lane<32>(sum) * 0x1p-24f;
}
__device__ __forceinline__ float output_factor(float l) { return (l > 0.f ? 1.0f / l : 0.f) * SPLIT_DOWN; }

// Four waves of 32 queries.  With the fp32 instruction 192 heads x 1024 x 64 took 383 us and 512 x 256 x 32 61 (now: beside the functions
// above); relative error against 64 bits at 4 x 512 x 64 1.9e-7 (fp32 instruction: 2.4e-7).  Vector issue bounds it, as in backward.
// Head sizes over 64 keep the fp32 instruction: their operands do not fit the registers in three parts.
template <int D>
__global__ __launch_bounds__(256, D > 64 ? 1 : 2) void k_flash_fwd_f32(FlashArgs a) {
  constexpr int EXACT = 2 * BC * (D + 1) * 4;
  int bh, xblk;
  flash_block(bh, xblk, flash_head_group(a.T, D, 4));
  xblk = gridDim.x - 1 - xblk;                                     // longest (latest) query blocks are scheduled first
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const int q0 = xblk * (WAVES * 32) + wave * 32, qi = q0 + lr, end = min(a.T, (xblk + 1) * (WAVES * 32));      // causal: keys < end
  if constexpr (D > 64) {
    __shared__ float smem[EXACT / 4];
    flash_fwd_exact<D>(a, bh, q0, end, true, smem);
  } else {
    using S = SplitTile<D>;
    __shared__ __attribute__((aligned(16))) char smem[2 * S::BYTES > EXACT ? 2 * S::BYTES : EXACT];
    char *Kr = smem, *Vc = smem + S::BYTES;
    const int b = bh / a.H, h = bh % a.H;
    const float *K = (const float *)a.k + b * a.k_sb + h * a.k_sh;
    const float *V = (const float *)a.v + b * a.v_sb + h * a.v_sh;
    const float factor = split_cap_factor(a.cap), mul = cap_mul(a);
    float qx[D / 16][8];
    S::row((const float *)a.q + b * a.q_sb + h * a.q_sh + (int64_t)qi * a.q_st, qi < a.T, a.hd, lk, qx);
    f32x16 o[S::F];
#pragma unroll
    for (int d = 0; d < S::F; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) o[d][e] = 0.f;
    float m = -INFINITY, l = 0.f;
    float kx[4][S::F], vx[4][S::F];
    S::load(kx, K, a.k_st, 0, a.T, a.hd);
    S::load(vx, V, a.v_st, 0, a.T, a.hd);
    bf16x8 q[D / 16][3];
    S::cut(qx, a.scale * SPLIT_UP, q);
    bool fine = split_cap_ok(a.cap);
    for (int kv0 = 0; kv0 < end; kv0 += BC) {
      S::scale(kx, SPLIT_UP);
      S::scale(vx, SPLIT_UP);
      __syncthreads();
      S::template put<true, false>(kx, Kr, nullptr);
      S::template put<false, true>(vx, nullptr, Vc);
      S::load(kx, K, a.k_st, kv0 + BC, a.T, a.hd);                 // the next tile, while this one is multiplied; rows past the end read as zero
      S::load(vx, V, a.v_st, kv0 + BC, a.T, a.hd);
      __syncthreads();
      if (kv0 > q0 + 31) continue;                                 // whole tile is in this wave's future (uniform per wave)
      f32x16 s;
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] = 0.f;
#pragma unroll
      for (int i = 0; i < D / 16; i++) {
        bf16x8 f[3];
        S::get_row(Kr, lr, 2 * i + lk, f);
        mfma6(f, q[i], s);
      }
      fine = fine && all_finite(s);
      const float top = tile_scores(s, a, factor, kv0, qi, lk);
      float alpha;
      const float sum = tile_weights(s, mul, m, top, alpha);
      l = __builtin_fmaf(l, alpha, sum);
      m = fmaxf(m, top);
      S::contract_rows(Vc, s, lr, lk, alpha, o);
    }
    fine = __all(fine && all_finite<S::F>(o));
    if (fine && qi < a.T) {
      const float f = output_factor(l);
      float *O = (float *)a.o + b * a.o_sb + h * a.o_sh + (int64_t)qi * a.o_st;
#pragma unroll
      for (int d = 0; d < S::F; d++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (32 * d + 8 * j + 4 * lk < a.hd)
            *reinterpret_cast<float4 *>(O + 32 * d + 8 * j + 4 * lk) = make_float4(o[d][4 * j] * f, o[d][4 * j + 1] * f, o[d][4 * j + 2] * f, o[d][4 * j + 3] * f);
      if (lk == 0) a.lse[((int64_t)b * a.H + h) * a.T + qi] = m + logf(l);
    }
    if (__syncthreads_or(!fine)) flash_fwd_exact<D>(a, bh, q0, end, !fine, (float *)smem);
  }
}

// The same for few blocks of 128 queries, where the chain of T / 32 tiles one after the other on a few CUs bounds the kernel above: a
// block owns 32 queries, and its 8 waves take 8 tiles at a time.  Each has its tile's scores, K and V straight from memory in the
// operand registers; the waves tell one another their columns' largest scores, so that each weighs its tile against the largest
// up to it, as the kernel above does; and the 8 products are added up in LDS in the order of the tiles, a thread holding two
// features of a query from each 32.  12 heads x 500 x 64: 61 us by the kernel above, 23 here (36 with sums of its own for every wave, by
// the fp32 instruction, whose last bits then depended on the number of heads); x 1024: 118, 61 (95); x 64: 11.7, 9.8.
template <int D>
__global__ __launch_bounds__(512, 2) void k_flash_fwd_f32_keys(FlashArgs a) {
  using S = SplitTile<D>;
  constexpr int W = 8, EXACT = 2 * BC * (D + 1) * 4, PART = W * 4096;
  __shared__ __attribute__((aligned(16))) char smem[PART > EXACT ? PART : EXACT];
  __shared__ float Top[W * 32], Alpha[W * 32], Sum[W * 32];
  int bh, xblk;
  flash_block(bh, xblk, flash_head_group(a.T, D, 4));
  xblk = gridDim.x - 1 - xblk;                                     // longest (latest) query blocks are scheduled first
  const int b = bh / a.H, h = bh % a.H;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const int q0 = xblk * 32, qi = q0 + lr, tiles = xblk + 1;
  const int r = threadIdx.x >> 4, c = threadIdx.x & 15;            // the sums: query q0 + r, features 2 c and 2 c + 1 of each 32
  const float *K = (const float *)a.k + b * a.k_sb + h * a.k_sh;
  const float *V = (const float *)a.v + b * a.v_sb + h * a.v_sh;
  const float factor = split_cap_factor(a.cap), mul = cap_mul(a);
  float qx[D / 16][8], k[D / 16][8], v[S::F][16];
  S::row((const float *)a.q + b * a.q_sb + h * a.q_sh + (int64_t)qi * a.q_st, qi < a.T, a.hd, lk, qx);
  auto load = [&](int i) {                                         // rows past the end read as zero
    if (i >= tiles) return;
    S::row(K + (int64_t)(32 * i + lr) * a.k_st, 32 * i + lr < a.T, a.hd, lk, k);
#pragma unroll
    for (int d = 0; d < S::F; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int kv = 32 * i + 8 * (e >> 2) + 4 * lk + (e & 3);
        v[d][e] = kv < a.T && 32 * d + lr < a.hd ? V[(int64_t)kv * a.v_st + 32 * d + lr] : 0.f;
      }
  };
  float o[S::F][2], m = -INFINITY, l = 0.f;                        // m of query qi, l of query q0 + r
#pragma unroll
  for (int d = 0; d < S::F; d++) o[d][0] = o[d][1] = 0.f;
  bool fine = split_cap_ok(a.cap);
  load(wave);
  bf16x8 q[D / 16][3];
  S::cut(qx, a.scale * SPLIT_UP, q);
  for (int first = 0; first < tiles; first += W) {
    const int i = first + wave;
    f32x16 s, t[S::F];
    float top = -INFINITY;
    if (i < tiles) {
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] = 0.f;
#pragma unroll
      for (int u = 0; u < D / 16; u++) {
        bf16x8 f[3];
#pragma unroll
        for (int e = 0; e < 8; e++) k[u][e] = here(k[u][e]) * SPLIT_UP;
        split8(k[u], f);
        mfma6(f, q[u], s);
      }
      fine = fine && all_finite(s);
      top = tile_scores(s, a, factor, 32 * i, qi, lk);
    }
    if (lk == 0) Top[wave * 32 + lr] = top;
    __syncthreads();
    float before = m;                                              // the largest score ahead of this wave's tile
#pragma unroll
    for (int w = 0; w < W; w++) {
      const float x = Top[w * 32 + lr];
      m = fmaxf(m, x);
      if (w < wave) before = fmaxf(before, x);
    }
    if (i < tiles) {
      float alpha;
      const float sum = tile_weights(s, mul, before, top, alpha);
      if (lk == 0) { Alpha[wave * 32 + lr] = alpha; Sum[wave * 32 + lr] = sum; }
      bf16x8 p[2][3];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const float x[8] = {s[8 * j], s[8 * j + 1], s[8 * j + 2], s[8 * j + 3], s[8 * j + 4], s[8 * j + 5], s[8 * j + 6], s[8 * j + 7]};
        split8(x, p[j]);
      }
#pragma unroll
      for (int d = 0; d < S::F; d++) {
#pragma unroll
        for (int e = 0; e < 16; e++) t[d][e] = 0.f;
#pragma unroll
        for (int j = 0; j < 2; j++) {
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; e++) x[e] = here(v[d][8 * j + e]) * SPLIT_UP;
          bf16x8 f[3];
          split8(x, f);
          mfma6(f, p[j], t[d]);
        }
      }
    }
    load(i + W);
    // features 4 g .. 4 g + 3 of a query are 16 bytes, in a row of 32 queries turned by 4 g: neither side meets a bank twice
#pragma unroll
    for (int d = 0; d < S::F; d++) {
      if (d) __syncthreads();
      if (i < tiles) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int g = 2 * j + lk;
          *reinterpret_cast<float4 *>(smem + ((wave * 8 + g) * 32 + ((lr + 4 * g) & 31)) * 16) = make_float4(t[d][4 * j], t[d][4 * j + 1], t[d][4 * j + 2], t[d][4 * j + 3]);
        }
      }
      __syncthreads();
      const int g = c >> 1;
      for (int w = 0; w < min(W, tiles - first); w++) {
        const float alpha = Alpha[w * 32 + r];
        const float2 x = *reinterpret_cast<const float2 *>(smem + ((w * 8 + g) * 32 + ((r + 4 * g) & 31)) * 16 + 8 * (c & 1));
        if (d == 0) l = __builtin_fmaf(l, alpha, Sum[w * 32 + r]);
        o[d][0] = __builtin_fmaf(o[d][0], alpha, x.x);
        o[d][1] = __builtin_fmaf(o[d][1], alpha, x.y);
      }
    }
  }
  float z = 0.f;
#pragma unroll
  for (int d = 0; d < S::F; d++) z = __builtin_fmaf(o[d][0], 0.f, __builtin_fmaf(o[d][1], 0.f, z));      // 0 unless one is infinite or NaN
  if (__syncthreads_or(!fine || !(z == 0.f))) {
    flash_fwd_exact<D>(a, bh, q0, min(a.T, q0 + 32), wave == 0, (float *)smem);
    return;
  }
  if (q0 + r < a.T) {
    const float f = output_factor(l);
    float *O = (float *)a.o + b * a.o_sb + h * a.o_sh + (int64_t)(q0 + r) * a.o_st;
#pragma unroll
    for (int d = 0; d < S::F; d++)
      if (32 * d + 2 * c < a.hd) *reinterpret_cast<float2 *>(O + 32 * d + 2 * c) = make_float2(o[d][0] * f, o[d][1] * f);
  }
  if (c == 0) Sum[r] = l;
  __syncthreads();
  if (threadIdx.x < 32 && qi < a.T) a.lse[((int64_t)b * a.H + h) * a.T + qi] = m + logf(Sum[lr]);
}

// delta[b,h,t] = sum_d dO[t,d] * O[t,d]: D / 4 lanes to a row of D features, 16 bytes each (a wave to a row, 4 bytes each, half of its
// lanes without any at head size 32, took 31 us for 512 heads x 256 x 32 and 44 us for 192 x 1024 x 64)
template <int D>
__global__ __launch_bounds__(256) void k_flash_delta_f32(FlashArgs a) {
  constexpr int L = D / 4;
  const int64_t row = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / L, total = (int64_t)a.B * a.H * a.T;
  const int d = 4 * (threadIdx.x % L);
  float s = 0.f;
  if (row < total && d < a.hd) {
    const int t = (int)(row % a.T), h = (int)((row / a.T) % a.H), b = (int)(row / ((int64_t)a.T * a.H));
    const int64_t at = b * a.o_sb + h * a.o_sh + (int64_t)t * a.o_st + d;
    const float4 o = *reinterpret_cast<const float4 *>((const float *)a.o + at), g = *reinterpret_cast<const float4 *>((const float *)a.d_o + at);
    s = __builtin_fmaf(o.x, g.x, o.y * g.y) + __builtin_fmaf(o.z, g.z, o.w * g.w);
  }
  s = near_sum<L>(s);
  if (row < total && d == 0) a.delta[row] = s;
}

// ------------------------------------------------------------------------------------------ dQ
template <int D>
__device__ void flash_dq_exact(const FlashArgs &a, int bh, int xblk, float *smem) {
  constexpr int P = D + 1, DB = D / 32;
  float *Ks = smem, *Vs = Ks + BC * P;
  int b = bh / a.H, h = bh % a.H;
  int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  int q0 = xblk * (WAVES * 32) + wave * 32, qi = q0 + lr;
  const float *Q = (const float *)a.q + b * a.q_sb + h * a.q_sh;
  const float *K = (const float *)a.k + b * a.k_sb + h * a.k_sh;
  const float *V = (const float *)a.v + b * a.v_sb + h * a.v_sh;
  const float *dO = (const float *)a.d_o + b * a.o_sb + h * a.o_sh;
  const float inv_cap = inverse_cap(a.cap);
  bool live = qi < a.T;
  float qreg[D / 2], doreg[D / 2];
#pragma unroll
  for (int i = 0; i < D / 2; i++) {
    qreg[i] = live && 2 * i + lk < a.hd ? Q[(int64_t)qi * a.q_st + 2 * i + lk] * a.scale : 0.f;
    doreg[i] = live && 2 * i + lk < a.hd ? dO[(int64_t)qi * a.o_st + 2 * i + lk] : 0.f;
  }
  int64_t srow = ((int64_t)b * a.H + h) * a.T + qi;
  float lse = live ? a.lse[srow] : 0.f, delta = live ? a.delta[srow] : 0.f;

  f32x16 dq[DB];
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int e = 0; e < 16; e++) dq[d][e] = 0.f;

  int q_block_end = min(a.T, (xblk + 1) * (WAVES * 32));
  for (int kv0 = 0; kv0 < q_block_end; kv0 += BC) {
    __syncthreads();
    load_tile_f32<D>(Ks, K, a.k_st, kv0, a.T, 1.0f, a.hd);
    load_tile_f32<D>(Vs, V, a.v_st, kv0, a.T, 1.0f, a.hd);
    __syncthreads();
    if (kv0 > q0 + 31) continue;
    f32x16 s, dp;
#pragma unroll
    for (int e = 0; e < 16; e++) { s[e] = 0.f; dp[e] = 0.f; }
#pragma unroll
    for (int i = 0; i < D / 2; i++) {
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(Ks[lr * P + 2 * i + lk], qreg[i], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(Vs[lr * P + 2 * i + lk], doreg[i], dp, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 16; e++) {
      int kv = kv0 + 8 * (e >> 2) + 4 * lk + (e & 3);
      float slope, sc = softcap_both(s[e], a.cap, inv_cap, slope);
      float p = (kv > qi || kv >= a.T || !live) ? 0.f : expf(sc - lse);
      s[e] = p * (dp[e] - delta) * slope * a.scale;
    }
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) {
        int kvr = 8 * (e >> 2) + 4 * lk + (e & 3);
        dq[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(Ks[kvr * P + 32 * d + lr], s[e], dq[d], 0, 0, 0);
      }
  }
  if (live) {
    float *dQ = (float *)a.dq + b * a.q_sb + h * a.q_sh + (int64_t)qi * a.q_st;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (32 * d + 8 * j + 4 * lk < a.hd)
          *reinterpret_cast<float4 *>(dQ + 32 * d + 8 * j + 4 * lk) = make_float4(dq[d][4 * j], dq[d][4 * j + 1], dq[d][4 * j + 2], dq[d][4 * j + 3]);
  }
}

template <int D>
__global__ __launch_bounds__(256, D > 64 ? 1 : 2) void k_flash_dq_f32(FlashArgs a) {
  constexpr int EXACT = 2 * BC * (D + 1) * 4;
  int bh, xblk;
  flash_block(bh, xblk, flash_head_group(a.T, D, 4));
  xblk = gridDim.x - 1 - xblk;                                     // longest (latest) query blocks are scheduled first
  if constexpr (D > 64) {
    __shared__ float smem[EXACT / 4];
    flash_dq_exact<D>(a, bh, xblk, smem);
  } else {
    using S = SplitTile<D>;
    __shared__ __attribute__((aligned(16))) char smem[3 * S::BYTES > EXACT ? 3 * S::BYTES : EXACT];
    char *Kr = smem, *Kc = smem + S::BYTES, *Vr = smem + 2 * S::BYTES;
    const int b = bh / a.H, h = bh % a.H;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
    const int q0 = xblk * (WAVES * 32) + wave * 32, qi = q0 + lr;
    const float *K = (const float *)a.k + b * a.k_sb + h * a.k_sh;
    const float *V = (const float *)a.v + b * a.v_sb + h * a.v_sh;
    // a score is mul times what scores_tanh leaves, t, and its derivative 1 - slope t^2
    const float factor = split_cap_factor(a.cap), mul = cap_mul(a), slope = a.cap > 0.f ? 1.0f : 0.f;
    const bool live = qi < a.T;
    float qx[D / 16][8], gx[D / 16][8];
    S::row((const float *)a.q + b * a.q_sb + h * a.q_sh + (int64_t)qi * a.q_st, live, a.hd, lk, qx);
    S::row((const float *)a.d_o + b * a.o_sb + h * a.o_sh + (int64_t)qi * a.o_st, live, a.hd, lk, gx);
    const int64_t srow = ((int64_t)b * a.H + h) * a.T + qi;
    const float lse = live ? a.lse[srow] : 0.f, delta = live ? a.delta[srow] : 0.f;
    f32x16 dq[S::F];
#pragma unroll
    for (int d = 0; d < S::F; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) dq[d][e] = 0.f;
    const int end = min(a.T, (xblk + 1) * (WAVES * 32));
    float kx[4][S::F], vx[4][S::F];
    S::load(kx, K, a.k_st, 0, a.T, a.hd);
    S::load(vx, V, a.v_st, 0, a.T, a.hd);
    bf16x8 q[D / 16][3], go[D / 16][3];
    S::cut(qx, a.scale * SPLIT_UP, q);
    S::cut(gx, SPLIT_UP, go);
    bool fine = split_cap_ok(a.cap);
    for (int kv0 = 0; kv0 < end; kv0 += BC) {
      S::scale(kx, SPLIT_UP);
      S::scale(vx, SPLIT_UP);
      __syncthreads();
      S::template put<true, true>(kx, Kr, Kc);
      S::template put<true, false>(vx, Vr, nullptr);
      S::load(kx, K, a.k_st, kv0 + BC, a.T, a.hd);                 // the next tile, while this one is multiplied; rows past the end read as zero
      S::load(vx, V, a.v_st, kv0 + BC, a.T, a.hd);
      __syncthreads();
      if (kv0 > q0 + 31) continue;                                 // whole tile is in this wave's future (uniform per wave)
      f32x16 s, dp;
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] = dp[e] = 0.f;
#pragma unroll
      for (int i = 0; i < D / 16; i++) {
        bf16x8 f[3];
        S::get_row(Kr, lr, 2 * i + lk, f);
        mfma6(f, q[i], s);
        S::get_row(Vr, lr, 2 * i + lk, f);
        mfma6(f, go[i], dp);
      }
      fine = fine && scores_finite(s);
      scores_tanh(s, a.cap, factor);
      auto weigh = [&](auto masks) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int kv = kv0 + 8 * (e >> 2) + 4 * lk + (e & 3);
          const float t = s[e];
          float p = exp_of<0>(__builtin_fmaf(t, mul, -lse));
          if (decltype(masks)::value) p = kv > qi || kv >= a.T || !live ? 0.f : p;
          const float ds = p * __builtin_fmaf(dp[e], SPLIT_DOWN, -delta) * __builtin_fmaf(-(t * slope), t, 1.0f);
          s[e] = ds * (a.scale * SPLIT_UP);
        }
      };
      if (__all(live && kv0 + 31 <= qi && kv0 + 32 <= a.T)) weigh(std::false_type());
      else weigh(std::true_type());
      S::contract_rows(Kc, s, lr, lk, 1.0f, dq);
    }
    if (__syncthreads_or(!fine || !all_finite<S::F>(dq))) {
      flash_dq_exact<D>(a, bh, xblk, (float *)smem);
      return;
    }
    if (live) {
      float *dQ = (float *)a.dq + b * a.q_sb + h * a.q_sh + (int64_t)qi * a.q_st;
#pragma unroll
      for (int d = 0; d < S::F; d++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (32 * d + 8 * j + 4 * lk < a.hd)
            *reinterpret_cast<float4 *>(dQ + 32 * d + 8 * j + 4 * lk) = summed(dq[d], j);
    }
  }
}

// ------------------------------------------------------------------------------------------ dK, dV
template <int D>
__device__ void flash_dkv_exact(const FlashArgs &a, int bh, int xblk, float *smem) {
  constexpr int P = D + 1, DB = D / 32;
  float *Qs = smem, *dOs = Qs + BC * P, *Ls = dOs + BC * P, *Ds = Ls + BC;
  int b = bh / a.H, h = bh % a.H;
  int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  int kv_blk0 = xblk * (WAVES * 32), kv0 = kv_blk0 + wave * 32, kvi = kv0 + lr;
  const float *Q = (const float *)a.q + b * a.q_sb + h * a.q_sh;
  const float *K = (const float *)a.k + b * a.k_sb + h * a.k_sh;
  const float *V = (const float *)a.v + b * a.v_sb + h * a.v_sh;
  const float *dO = (const float *)a.d_o + b * a.o_sb + h * a.o_sh;
  const float inv_cap = inverse_cap(a.cap);
  bool live = kvi < a.T;
  float kreg[D / 2], vreg[D / 2];
#pragma unroll
  for (int i = 0; i < D / 2; i++) {
    kreg[i] = live && 2 * i + lk < a.hd ? K[(int64_t)kvi * a.k_st + 2 * i + lk] : 0.f;
    vreg[i] = live && 2 * i + lk < a.hd ? V[(int64_t)kvi * a.v_st + 2 * i + lk] : 0.f;
  }
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int e = 0; e < 16; e++) { dk[d][e] = 0.f; dv[d][e] = 0.f; }

  int64_t srow0 = ((int64_t)b * a.H + h) * a.T;
  for (int q0 = kv_blk0; q0 < a.T; q0 += BC) {        // causal: queries at or after this block's first key
    __syncthreads();
    load_tile_f32<D>(Qs, Q, a.q_st, q0, a.T, a.scale, a.hd);
    load_tile_f32<D>(dOs, dO, a.o_st, q0, a.T, 1.0f, a.hd);
    if (threadIdx.x < BC) {
      int qi = q0 + threadIdx.x;
      Ls[threadIdx.x] = qi < a.T ? a.lse[srow0 + qi] : 0.f;
      Ds[threadIdx.x] = qi < a.T ? a.delta[srow0 + qi] : 0.f;
    }
    __syncthreads();
    if (q0 + 31 < kv0) continue;                      // every query of the tile precedes this wave's keys
    f32x16 s, dp;
#pragma unroll
    for (int e = 0; e < 16; e++) { s[e] = 0.f; dp[e] = 0.f; }
#pragma unroll
    for (int i = 0; i < D / 2; i++) {                 // rows = queries, columns = this wave's keys
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(Qs[lr * P + 2 * i + lk], kreg[i], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(dOs[lr * P + 2 * i + lk], vreg[i], dp, 0, 0, 0);
    }
    f32x16 pm;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      int qr = 8 * (e >> 2) + 4 * lk + (e & 3), qi = q0 + qr;
      float slope, sc = softcap_both(s[e], a.cap, inv_cap, slope);
      float p = (kvi > qi || qi >= a.T || !live) ? 0.f : expf(sc - Ls[qr]);
      pm[e] = p;
      s[e] = p * (dp[e] - Ds[qr]) * slope;                                      // Qs already carries `scale`, so dK = dS^T (scale*Q)
    }
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) {
        int qr = 8 * (e >> 2) + 4 * lk + (e & 3);
        dv[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(dOs[qr * P + 32 * d + lr], pm[e], dv[d], 0, 0, 0);
        dk[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(Qs[qr * P + 32 * d + lr], s[e], dk[d], 0, 0, 0);
      }
  }
  if (live) {
    float *dK = (float *)a.dk + b * a.k_sb + h * a.k_sh + (int64_t)kvi * a.k_st;
    float *dV = (float *)a.dv + b * a.v_sb + h * a.v_sh + (int64_t)kvi * a.v_st;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (32 * d + 8 * j + 4 * lk >= a.hd) continue;
        *reinterpret_cast<float4 *>(dK + 32 * d + 8 * j + 4 * lk) = make_float4(dk[d][4 * j], dk[d][4 * j + 1], dk[d][4 * j + 2], dk[d][4 * j + 3]);
        *reinterpret_cast<float4 *>(dV + 32 * d + 8 * j + 4 * lk) = make_float4(dv[d][4 * j], dv[d][4 * j + 1], dv[d][4 * j + 2], dv[d][4 * j + 3]);
      }
  }
}

template <int D>
__global__ __launch_bounds__(256, D > 64 ? 1 : 2) void k_flash_dkv_f32(FlashArgs a) {
  constexpr int EXACT = (2 * BC * (D + 1) + 2 * BC) * 4;
  int bh, xblk;
  flash_block(bh, xblk, flash_head_group(a.T, D, 4));
  if constexpr (D > 64) {
    __shared__ float smem[EXACT / 4];
    flash_dkv_exact<D>(a, bh, xblk, smem);
  } else {
    using S = SplitTile<D>;
    constexpr int LDS = 4 * S::BYTES + 2 * BC * 4;
    __shared__ __attribute__((aligned(16))) char smem[LDS > EXACT ? LDS : EXACT];
    char *Qr = smem, *Qc = smem + S::BYTES, *Gr = smem + 2 * S::BYTES, *Gc = smem + 3 * S::BYTES;
    float *Ls = (float *)(smem + 4 * S::BYTES), *Ds = Ls + BC;
    const int b = bh / a.H, h = bh % a.H;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
    const int kv_blk0 = xblk * (WAVES * 32), kv0 = kv_blk0 + wave * 32, kvi = kv0 + lr;
    const float *Q = (const float *)a.q + b * a.q_sb + h * a.q_sh;
    const float *dO = (const float *)a.d_o + b * a.o_sb + h * a.o_sh;
    const float factor = split_cap_factor(a.cap), mul = cap_mul(a), slope = a.cap > 0.f ? 1.0f : 0.f;      // as in dQ
    const bool live = kvi < a.T;
    // K's and V's rows stay whole and are cut where they are used: in three parts, they, the accumulators and the next tile are more
    // registers than a wave of two per SIMD has (the empty assembler statements keep the cuts from being moved out of the loop).
    float k[D / 16][8], v[D / 16][8];
    S::row((const float *)a.k + b * a.k_sb + h * a.k_sh + (int64_t)kvi * a.k_st, live, a.hd, lk, k);
    S::row((const float *)a.v + b * a.v_sb + h * a.v_sh + (int64_t)kvi * a.v_st, live, a.hd, lk, v);
    f32x16 dk[S::F], dv[S::F];
#pragma unroll
    for (int d = 0; d < S::F; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) { dk[d][e] = 0.f; dv[d][e] = 0.f; }
    const int64_t srow0 = ((int64_t)b * a.H + h) * a.T;
    float qx[4][S::F], gx[4][S::F], stat = 0.f;
    auto load = [&](int q0) {
      S::load(qx, Q, a.q_st, q0, a.T, a.hd);
      S::load(gx, dO, a.o_st, q0, a.T, a.hd);
      const int qi = q0 + (threadIdx.x & 31);
      if (threadIdx.x < 64) stat = qi < a.T ? (threadIdx.x < 32 ? a.lse : a.delta)[srow0 + qi] : 0.f;
    };
    load(kv_blk0);
    S::scale(k, SPLIT_UP);
    S::scale(v, SPLIT_UP);
    float top = 0.f;
#pragma unroll
    for (int i = 0; i < D / 16; i++)
#pragma unroll
      for (int e = 0; e < 8; e += 2) top = fmaxf(fmaxf(top, fabsf(k[i][e])), fabsf(k[i][e + 1]));
    bool fine = split_cap_ok(a.cap) && top < LARGE_OPERAND * SPLIT_UP;
    for (int q0 = kv_blk0; q0 < a.T; q0 += BC) {                   // causal: queries at or after this block's first key
      S::scale(qx, a.scale * SPLIT_UP);
      S::scale(gx, SPLIT_UP);
      fine = fine && S::largest(qx) < LARGE_OPERAND * SPLIT_UP;
      __syncthreads();
      S::template put<true, true>(qx, Qr, Qc);
      S::template put<true, true>(gx, Gr, Gc);
      if (threadIdx.x < 64) Ls[threadIdx.x] = stat;                // the second 32 are Ds
      load(q0 + BC);                                               // the next tile, while this one is multiplied; rows past the end read as zero
      __syncthreads();
      if (q0 + 31 < kv0) continue;                                 // every query of the tile precedes this wave's keys
      f32x16 s, dp;
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] = dp[e] = 0.f;
#pragma unroll
      for (int i = 0; i < D / 16; i++) {                           // rows = queries, columns = this wave's keys
        bf16x8 f[3];
        S::get_row(Qr, lr, 2 * i + lk, f);
        bf16x8 u[3], w[3];
#pragma unroll
        for (int e = 0; e < 8; e++) asm volatile("" : "+v"(k[i][e]), "+v"(v[i][e]));
        split8(k[i], u);
        split8(v[i], w);
        mfma6(f, u, s);
        S::get_row(Gr, lr, 2 * i + lk, f);
        mfma6(f, w, dp);
      }
      f32x16 pm;
      scores_tanh(s, a.cap, factor);
      auto weigh = [&](auto masks) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int qr = 8 * (e >> 2) + 4 * lk + (e & 3), qi = q0 + qr;
          const float t = s[e];
          float p = exp_of<24>(__builtin_fmaf(t, mul, -Ls[qr]));
          if (decltype(masks)::value) p = kvi > qi || qi >= a.T || !live ? 0.f : p;
          pm[e] = p;
          // Qc already carries `scale`, so dK = dS^T (scale*Q)
          s[e] = p * __builtin_fmaf(dp[e], SPLIT_DOWN, -Ds[qr]) * __builtin_fmaf(-(t * slope), t, 1.0f);
        }
      };
      if (__all(live && kvi <= q0 && q0 + 32 <= a.T)) weigh(std::false_type());
      else weigh(std::true_type());
      S::contract_rows(Gc, pm, lr, lk, 1.0f, dv);
      S::contract_rows(Qc, s, lr, lk, 1.0f, dk);
    }
    if (__syncthreads_or(!fine || !all_finite<S::F>(dk) || !all_finite<S::F>(dv))) {
      flash_dkv_exact<D>(a, bh, xblk, (float *)smem);
      return;
    }
    if (live) {
      float *dK = (float *)a.dk + b * a.k_sb + h * a.k_sh + (int64_t)kvi * a.k_st;
      float *dV = (float *)a.dv + b * a.v_sb + h * a.v_sh + (int64_t)kvi * a.v_st;
#pragma unroll
      for (int d = 0; d < S::F; d++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          if (32 * d + 8 * j + 4 * lk >= a.hd) continue;
          *reinterpret_cast<float4 *>(dK + 32 * d + 8 * j + 4 * lk) = summed(dk[d], j);
          *reinterpret_cast<float4 *>(dV + 32 * d + 8 * j + 4 * lk) = summed(dv[d], j);
        }
    }
  }
}

int32_t check(const AhFlash *f, bool bwd, FlashArgs &a) {
  AH_ARG(f != nullptr, "flash attention: null descriptor");
  AH_ARG(f->dtype == AH_F32 || f->dtype == AH_BF16, "flash attention: dtype %d must be f32 or bf16", f->dtype);
  AH_ARG(f->head_dim >= 8 && f->head_dim <= 128 && f->head_dim % 8 == 0, "flash attention: head_dim %d is not a multiple of 8 from 8 to 128", f->head_dim);
  AH_ARG(f->batch >= 0 && f->heads >= 0 && f->seq >= 0, "flash attention: negative extent");
  AH_ARG((int64_t)f->batch * f->heads <= 65535, "flash attention: batch*heads %lld exceeds 65535", (long long)f->batch * f->heads);
  AH_ARG(f->q && f->k && f->v && f->o && f->lse, "flash attention: null operand");
  const int64_t st[] = {f->q_sb, f->q_sh, f->q_st, f->k_sb, f->k_sh, f->k_st, f->v_sb, f->v_sh, f->v_st, f->o_sb, f->o_sh, f->o_st};
  const int64_t sm = f->dtype == AH_BF16 ? 8 : 4;        // rows are moved in 16-byte pieces
  for (int64_t s : st) AH_ARG(s % sm == 0 && s >= 0, "flash attention: strides must be non-negative multiples of 16 bytes");
  AH_ARG(f->q_st >= f->head_dim && f->k_st >= f->head_dim && f->v_st >= f->head_dim && f->o_st >= f->head_dim,
         "flash attention: row stride smaller than head_dim");
  AH_ARG(aligned16(f->q) && aligned16(f->k) && aligned16(f->v) && aligned16(f->o), "flash attention: operands must be 16-byte aligned");
  if (bwd) {
    AH_ARG(f->d_o && f->dq && f->dk && f->dv, "flash attention backward: null gradient operand");
    AH_ARG(aligned16(f->d_o) && aligned16(f->dq) && aligned16(f->dk) && aligned16(f->dv), "flash attention backward: operands must be 16-byte aligned");
  }
  a.q = dp<const void>(f->q); a.k = dp<const void>(f->k); a.v = dp<const void>(f->v);
  a.o = dp<void>(f->o); a.lse = dp<float>(f->lse);
  a.d_o = dp<const void>(f->d_o); a.dq = dp<void>(f->dq); a.dk = dp<void>(f->dk); a.dv = dp<void>(f->dv);
  a.delta = nullptr; a.variant = f->bwd_variant;
  a.B = f->batch; a.H = f->heads; a.T = f->seq; a.hd = f->head_dim;
  a.q_sb = f->q_sb; a.q_sh = f->q_sh; a.q_st = f->q_st;
  a.k_sb = f->k_sb; a.k_sh = f->k_sh; a.k_st = f->k_st;
  a.v_sb = f->v_sb; a.v_sh = f->v_sh; a.v_st = f->v_st;
  a.o_sb = f->o_sb; a.o_sh = f->o_sh; a.o_st = f->o_st;
  a.scale = f->scale; a.cap = f->soft_cap;
  return AH_OK;
}

template <int D>
int32_t run_fwd(const FlashArgs &a) {
  if constexpr (D <= 64) {
    // What the two take, as measured: a block of 128 queries 3.7 us for each tile of its chain, whatever else is on its CU (up to two), a CU
    // 10 us for every 8 tiles of 32 queries that share their keys (`eights` of them per head); a single tile has nobody to share with
    // (5 heads x 29 x 64 6.6 / 8.4).  us, blocks of 128 / keys among waves:
    //   D = 64, 12 heads: T = 64 11.7 / 9.8, 256 33 / 14.6, 500 61 / 23, 1024 118 / 61, 2048 232 / 158; T = 1024 24 heads 121 / 81, 32 heads 124 / 103,
    //   192 heads 305 / 571; T = 256 64 heads 35 / 25, 96 heads 36 / 37; 64 heads x 512 x 48 65 / 60; 160 heads x T = 100 20 / 28
    //   D = 32: 8 heads x T = 40 9.8 / 7.3, x T = 256 29 / 10; 64 x 128 16 / 8.8; 152 x 250 31 / 41; 2 x 2050 210 / 49
    // A row has the same bits from both, so a head's result does not depend on how many others are in the call.
    const int64_t tiles = cdiv(a.T, 32), whole = tiles / 8, eights = 4 * whole * (whole + 1) + tiles % 8 * (whole + 1);
    const int64_t heads = (int64_t)a.B * a.H;
    if (tiles > 1 && 26 * eights * heads <= 10 * num_cus() * tiles) {
      ah::launch_kernel(k_flash_fwd_f32_keys<D>, dim3((unsigned)tiles, (unsigned)heads), dim3(512), 0, a);
      AH_LAUNCH_CHECK();
      return AH_OK;
    }
  }
  dim3 grid((unsigned)cdiv(a.T, WAVES * 32), (unsigned)(a.B * a.H));
  ah::launch_kernel(k_flash_fwd_f32<D>, grid, dim3(256), 0, a);
  AH_LAUNCH_CHECK();
  return AH_OK;
}
template <int D>
int32_t run_bwd(FlashArgs &a) {
  int64_t rows = (int64_t)a.B * a.H * a.T;
  ah_ptr delta = 0;
  int32_t rc = ah_alloc((uint64_t)rows * 4, &delta);
  if (rc) return rc;
  a.delta = dp<float>(delta);
  ah::launch_kernel(k_flash_delta_f32<D>, dim3((unsigned)cdiv(rows * (D / 4), 256)), dim3(256), 0, a);
  AH_LAUNCH_CHECK();
  dim3 grid((unsigned)cdiv(a.T, WAVES * 32), (unsigned)(a.B * a.H));
  ah::launch_kernel(k_flash_dq_f32<D>, grid, dim3(256), 0, a);
  AH_LAUNCH_CHECK();
  ah::launch_kernel(k_flash_dkv_f32<D>, grid, dim3(256), 0, a);
  AH_LAUNCH_CHECK();
  return ah_free(delta);
}

}  // namespace

extern "C" {

int32_t ah_flash_fwd(const AhFlash *f) {
  AH_REQUIRE_READY();
  FlashArgs a;
  int32_t rc = check(f, false, a);
  if (rc) return rc;
  if (a.B * a.H == 0 || a.T == 0) return AH_OK;
  const int tile_d = f->head_dim <= 32 ? 32 : f->head_dim <= 64 ? 64 : 128;      // the kernels' head size: the features beyond head_dim are zeros
  if (f->dtype == AH_BF16) return flash_fwd_bf16(a, tile_d);
  switch (tile_d) {
    case 32: return run_fwd<32>(a);
    case 64: return run_fwd<64>(a);
    default: return run_fwd<128>(a);
  }
}

int32_t ah_flash_bwd(const AhFlash *f) {
  AH_REQUIRE_READY();
  FlashArgs a;
  int32_t rc = check(f, true, a);
  if (rc) return rc;
  if (a.B * a.H == 0 || a.T == 0) return AH_OK;
  const int tile_d = f->head_dim <= 32 ? 32 : f->head_dim <= 64 ? 64 : 128;
  if (f->dtype == AH_BF16) return flash_bwd_bf16(a, tile_d);
  switch (tile_d) {
    case 32: return run_bwd<32>(a);
    case 64: return run_bwd<64>(a);
    default: return run_bwd<128>(a);
  }
}

}  // extern "C"
