// fp32 products on the bf16 matrix pipes.
//
// Every operand value is cut, on its way to the matrix pipe, into three bf16 numbers, and a product is six of theirs (split_bf16.h):
// 2.7 times the rate of the fp32 instruction.  How the sums are kept as close to the 64-bit ones as that instruction's: S_FLUSH below.
// A workgroup that finds a result that is not finite computes its tile again with the fp32 instruction (f32_tile), whose result stands.
#include "gemm_common.h"
#include "split_bf16.h"
#include <cmath>
#include <type_traits>

using namespace ah;

namespace {

// ================================================================ a tile with the fp32 instruction
// LDS tiles are k-major: As[k][m], Bs[k][n]; a lane of the 32x32x2 MFMA reads As[2*kk + lane/32][m0 + lane%32].
constexpr int F_BK = 16, F_PAD = 4;

// A [rows x F_BK] tile of an operand in registers: a float4 per thread for every 64 rows, 4 consecutive k of one row.  The row and the
// quarter of the 16 k of a thread's i-th:
//   KCONTIG = true : memory is [row][k] (k contiguous), 4 threads side by side along a row
//   KCONTIG = false: memory is [k][row] (row contiguous), a wave along 64 rows
template <bool KCONTIG>
__device__ __forceinline__ int part_row(int i) { return (KCONTIG ? threadIdx.x >> 2 : threadIdx.x & 63) + 64 * i; }
template <bool KCONTIG>
__device__ __forceinline__ int part_k4() { return KCONTIG ? threadIdx.x & 3 : threadIdx.x >> 6; }
// TAIL: k from K on reads as zero.  VEC: the rows of a k-contiguous operand are 16-byte aligned.
// The tile's corner is a scalar address and the thread's part of it 32 bits (the rows of a tile span less than 4 GiB).
template <bool KCONTIG, bool VEC, bool TAIL>
__device__ __forceinline__ float4 load_part(const float *__restrict__ base, int64_t ld, int row0, int k0, int rows, int K, int i) {
  const int t = threadIdx.x, kw = KCONTIG ? 0 : __builtin_amdgcn_readfirstlane(part_k4<KCONTIG>()) * 4, last = rows - 1 - row0;
  const float *corner = KCONTIG ? base + (int64_t)row0 * ld + k0 : base + (int64_t)(k0 + kw) * ld + row0;
  const int r = min(part_row<KCONTIG>(i), last);      // rows past the end repeat the last one: their results are not stored
  if (KCONTIG) {
    const int k = k0 + (t & 3) * 4;
    const float *p = reinterpret_cast<const float *>(reinterpret_cast<const char *>(corner) + ((uint32_t)r * (uint32_t)ld + (t & 3) * 4) * 4u);
    if (TAIL) return make_float4(k < K ? p[0] : 0.f, k + 1 < K ? p[1] : 0.f, k + 2 < K ? p[2] : 0.f, k + 3 < K ? p[3] : 0.f);
    if (VEC) return *reinterpret_cast<const float4 *>(p);
    return make_float4(p[0], p[1], p[2], p[3]);
  }
  const int k = k0 + kw;
  const float *p0 = corner, *p1 = p0 + ld, *p2 = p1 + ld, *p3 = p2 + ld;
  if (TAIL) return make_float4(k < K ? p0[r] : 0.f, k + 1 < K ? p1[r] : 0.f, k + 2 < K ? p2[r] : 0.f, k + 3 < K ? p3[r] : 0.f);
  return make_float4(p0[(uint32_t)r], p1[(uint32_t)r], p2[(uint32_t)r], p3[(uint32_t)r]);
}
template <bool KCONTIG, int N, bool VEC, bool TAIL>
__device__ __forceinline__ void load_tile(const float *__restrict__ base, int64_t ld, int row0, int k0, int rows, int K, float4 (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; i++) v[i] = load_part<KCONTIG, VEC, TAIL>(base, ld, row0, k0, rows, K, i);
}

// Four results side by side: what the epilogue makes of them, 16-byte accesses where vec.  PLAIN: f32 results as they are;
// otherwise the epilogue and the type of C are chosen at run time (they are the same for the whole launch).
template <bool PLAIN>
__device__ __forceinline__ void finish4(const GemmArgs &g, int64_t cbase, int row, int col, float4 v, bool vec, int out_bf16) {
  if (PLAIN) { epilogue4<AH_EPI_NONE, float>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec); return; }
  switch (g.epi) {
    case AH_EPI_NONE:
      if (out_bf16) epilogue4<AH_EPI_NONE, uint16_t>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec);
      else epilogue4<AH_EPI_NONE, float>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec);
      break;
    case AH_EPI_ACCUM: epilogue4<AH_EPI_ACCUM, float>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec); break;
    case AH_EPI_RESIDUAL: epilogue4<AH_EPI_RESIDUAL, float>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec); break;
    case AH_EPI_GELU: epilogue4<AH_EPI_GELU, float>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec); break;
    case AH_EPI_GELU_GRAD: epilogue4<AH_EPI_GELU_GRAD, float>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec); break;
    case AH_EPI_MUL_AUX: epilogue4<AH_EPI_MUL_AUX, float>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec); break;
    default: epilogue4<AH_EPI_GELU_BWD, float>(g, cbase, row, col, v.x, v.y, v.z, v.w, vec);
  }
}
// A 32 x 32 accumulator of a transposed product (element e is n = 8*(e/4) + 4*(lane/32) + e%4, m = lane%32) in 4 KB of LDS, row by
// row, the 16-byte pieces of a row permuted so that neither side of the exchange meets a bank twice.
__device__ __forceinline__ void stage_tile(char *stage, const f32x16 &acc) {
  const int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
#pragma unroll
  for (int q = 0; q < 4; q++)
    *reinterpret_cast<float4 *>(stage + lr * 128 + (((2 * q + lk) ^ (lr & 7)) << 4)) = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
}
__device__ __forceinline__ float4 staged(const char *stage, int row, int chunk) { return *reinterpret_cast<const float4 *>(stage + row * 128 + ((chunk ^ (row & 7)) << 4)); }
// Stores one: through the wave's own 4 KB of LDS, so that 8 lanes write the 128 bytes of a row side by side.
template <bool PLAIN>
__device__ __forceinline__ void finish_tile(const GemmArgs &g, int64_t cbase, int row0, int col0, const f32x16 &acc, bool vec, int out_bf16, char *stage) {
  const int lane = threadIdx.x & 63, r = lane >> 3, ch = lane & 7;
  stage_tile(stage, acc);
  if (PLAIN) {
#pragma unroll
    for (int it = 0; it < 4; it++) finish4<true>(g, cbase, row0 + it * 8 + r, col0 + 4 * ch, staged(stage, it * 8 + r, ch), vec, 0);
  } else {
#pragma unroll 1
    for (int it = 0; it < 4; it++) finish4<false>(g, cbase, row0 + it * 8 + r, col0 + 4 * ch, staged(stage, it * 8 + r, ch), vec, out_bf16);
  }
}

// The BM x BN tile at (m0, n0) by v_mfma_f32_32x32x2_f32, 2 x 2 waves; smem holds 2 * F_BK * (BM + BN + 2 F_PAD) floats.
template <bool A_KC, bool B_KC, int BM, int BN, bool VEC>
__device__ __forceinline__ void f32_tile(const GemmArgs &g, const float *A, const float *B, int64_t cbase, int m0, int n0, bool vec_c, int out_bf16, float *smem) {
  constexpr int PA = BM + F_PAD, PB = BN + F_PAD, TM = BM / 64, TN = BN / 64, NA = BM / 64, NB = BN / 64;
  float *As = smem, *Bs = smem + 2 * F_BK * PA;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
  float4 ra[NA], rb[NB];
  auto store = [&](float *s, int pitch, int r, int k4, const float4 &v) {
    const int k = 4 * k4;
    s[(k + 0) * pitch + r] = v.x; s[(k + 1) * pitch + r] = v.y; s[(k + 2) * pitch + r] = v.z; s[(k + 3) * pitch + r] = v.w;
  };
  const int full = g.K / F_BK, nt = (g.K + F_BK - 1) / F_BK;
  auto load = [&](int kt) {
    if (kt < full) {
      load_tile<A_KC, NA, VEC, false>(A, g.lda, m0, kt * F_BK, g.M, g.K, ra);
      load_tile<B_KC, NB, VEC, false>(B, g.ldb, n0, kt * F_BK, g.N, g.K, rb);
    } else if (kt < nt) {
      load_tile<A_KC, NA, VEC, true>(A, g.lda, m0, kt * F_BK, g.M, g.K, ra);
      load_tile<B_KC, NB, VEC, true>(B, g.ldb, n0, kt * F_BK, g.N, g.K, rb);
    }
  };
  load(0);
  for (int kt = 0; kt < nt; kt++) {
    float *as = As + (kt & 1) * F_BK * PA, *bs = Bs + (kt & 1) * F_BK * PB;
#pragma unroll
    for (int i = 0; i < NA; i++) store(as, PA, part_row<A_KC>(i), part_k4<A_KC>(), ra[i]);
#pragma unroll
    for (int i = 0; i < NB; i++) store(bs, PB, part_row<B_KC>(i), part_k4<B_KC>(), rb[i]);
    load(kt + 1);                               // on its way while this one is multiplied
    __syncthreads();                            // the other buffer was last read before the previous barrier
#pragma unroll
    for (int kk = 0; kk < F_BK / 2; kk++) {
      float a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; i++) a[i] = as[(2 * kk + lk) * PA + wm + 32 * i + lr];
#pragma unroll
      for (int j = 0; j < TN; j++) b[j] = bs[(2 * kk + lk) * PB + wn + 32 * j + lr];
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j], a[i], acc[i][j], 0, 0, 0);      // C^T tiles
    }
  }
  __syncthreads();                              // the tiles have been read: their memory takes the results
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) finish_tile<false>(g, cbase, m0 + wm + 32 * i, n0 + wn + 32 * j, acc[i][j], vec_c, out_bf16, (char *)smem + wave * 4096);
}

// ================================================================ the split
// TM x TN accumulators (C^T orientation) += the six products, the smallest first; FIRST: = the six products
template <bool FIRST, int TM, int TN>
__device__ __forceinline__ void mfma6_tiles(const bf16x8 (&a)[3][TM], const bf16x8 (&b)[3][TN], f32x16 (&acc)[TM][TN]) {
  const f32x16 zero = {0.f};
#pragma unroll
  for (int p = 0; p < 6; p++)
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[SPLIT_B[p]][j], a[SPLIT_A[p]][i], FIRST && p == 0 ? zero : acc[i][j], 0, 0, 0);
}

// ================================================================ tiles through LDS
// 2 x 2 waves of 64 x 64 (or 32 x 32): 24 matrix instructions per step and wave, 768 cycles, against 92 vector instructions for the
// split and the long sums, which go into the gaps between them (sched_group_barrier, four to a gap: with 3 or 6 3 to 12 % slower).
// What bounds the large tiles: on zeros, where the clock does not fall, 16384 x 3072 x 768 takes 341 us, without the split 275; on
// standard normal operands the clock falls to 1.9 GHz and it takes 436 from the hundredth call on, 560 over the first ten (matrix pipes
// 49 % busy).  One tile on its way instead of two cost 5 % there, the 64 vector instructions more of a split by shifts and subtractions
// nothing in NT and NN and 5 % in TN.  Tiles of
// 128 x 64, and 128 x 128 on eight waves, are slower at every size tried (2 to 30 %).
// LDS: three planes of [row][16 k] bf16 per operand, 32 bytes a row, two buffers.  The 16-byte half of a row that holds k 0..7 is
// the first one in rows whose bit 3 is clear and the second one in the others: the fragment reads and the 8-byte writes of either
// operand order then spread over all banks.
constexpr int S_BK = 16;
// The matrix instruction cuts the terms it adds off at the last place of the largest: a long sum drifts towards zero (3e-11 of it per step
// where all terms are positive, more where a large one comes first) besides being rounded more coarsely the larger it gets.  So every
// S_FLUSH steps the accumulator is added, rounded to nearest, to a second one.  Relative error against 64 bits, terms of either sign,
// at K = 768 / 16384: 1.2e-7 / 2.0e-7; without the second accumulator 4.2e-7 / 2.1e-6; the fp32 instruction 5.0e-7 and, in slices of
// 512, 4.2e-7.  Flushing every 16 steps is 2 % faster and left the gradients of a 6 x 256 model 1.6 times as far from 64 bits as the
// fp32 instruction does; every 4 steps leaves them where they were.
constexpr int S_FLUSH = 4;
static_assert(S_FLUSH == 4, "the loop of k_gemm_f32_split is written for it");
__device__ __forceinline__ int plane_ofs(int row, int k4) { return row * 32 + ((((k4 >> 1) ^ (row >> 3)) & 1) << 4) + (k4 & 1) * 8; }

template <bool KCONTIG, int ROWS, bool TAIL>
__device__ __forceinline__ void store_part(char *s, const float4 &v, int i) {
  const float4 x = TAIL ? make_float4(here(v.x), here(v.y), here(v.z), here(v.w)) : v;
  const Split2 a = split2(x.x * SPLIT_UP, x.y * SPLIT_UP), b = split2(x.z * SPLIT_UP, x.w * SPLIT_UP);
  char *p = s + plane_ofs(part_row<KCONTIG>(i), part_k4<KCONTIG>());
  *reinterpret_cast<uint2 *>(p) = make_uint2(a.h, b.h);
  *reinterpret_cast<uint2 *>(p + ROWS * 32) = make_uint2(a.m, b.m);
  *reinterpret_cast<uint2 *>(p + 2 * ROWS * 32) = make_uint2(a.l, b.l);
}
template <bool KCONTIG, int ROWS, bool TAIL>
__device__ __forceinline__ void store_split(char *s, const float4 (&v)[ROWS / 64]) {
#pragma unroll
  for (int i = 0; i < ROWS / 64; i++) store_part<KCONTIG, ROWS, TAIL>(s, v[i], i);
}
template <int ROWS, int T>
__device__ __forceinline__ void read_split(const char *s, int row0, int lr, int lk, bf16x8 (&f)[3][T]) {
#pragma unroll
  for (int p = 0; p < 3; p++)
#pragma unroll
    for (int i = 0; i < T; i++)
      f[p][i] = *reinterpret_cast<const bf16x8 *>(s + p * ROWS * 32 + (row0 + 32 * i + lr) * 32 + ((lk ^ (lr >> 3)) & 1) * 16);
}

// Which tile a workgroup takes: an XCD (workgroups are dealt to the eight in turn) takes a contiguous stretch of the tiles,
// in bands of 8 tile rows, so that the operand panels it reads again are in its own L2.
__device__ __forceinline__ void tile_of(int bid, int tiles_m, int tiles_n, int &tm, int &tn) {
  const int nb = tiles_m * tiles_n, xcd = bid & 7, q = nb >> 3, r = nb & 7;
  const int lin = xcd * q + min(xcd, r) + (bid >> 3);
  const int band = lin / (8 * tiles_n), first = band * 8, h = min(8, tiles_m - first), in = lin - first * tiles_n;
  tm = first + in % h;
  tn = in / h;
}

template <int LAYOUT, int BM, int BN, bool PLAIN, bool VEC>
__global__ __launch_bounds__(256, 2) void k_gemm_f32_split(GemmArgs g, int vec_c, int out_bf16) {
  constexpr bool A_KC = (LAYOUT != AH_GEMM_TN);     // A is [M][K] except for TN ([K][M])
  constexpr bool B_KC = (LAYOUT == AH_GEMM_NT);     // B is [N][K] only for NT
  constexpr int TM = BM / 64, TN = BN / 64, NA = BM / 64, NB = BN / 64;
  constexpr int ABYTES = 3 * BM * 32, BBYTES = 3 * BN * 32;
  constexpr int SPLIT_LDS = 2 * (ABYTES + BBYTES), F32_LDS = 2 * F_BK * (BM + BN + 2 * F_PAD) * 4;
  __shared__ __attribute__((aligned(16))) char smem[SPLIT_LDS > F32_LDS ? SPLIT_LDS : F32_LDS];
  const float *A = (const float *)g.a + (int64_t)blockIdx.z * g.sa;
  const float *B = (const float *)g.b + (int64_t)blockIdx.z * g.sb;
  const int64_t cbase = (int64_t)blockIdx.z * g.sc;
  if (g.nsplit > 1) g.K = min(g.ksplit, g.K - (int)blockIdx.z * g.ksplit);      // the batch entries are slices of one contraction
  int tm, tn;
  tile_of(blockIdx.x, (g.M + BM - 1) / BM, (g.N + BN - 1) / BN, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);

  f32x16 acc[TM][TN], sum[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = sum[i][j][e] = 0.f;
  auto flush = [&]() {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) sum[i][j][e] = __builtin_fmaf(acc[i][j][e], SPLIT_DOWN, sum[i][j][e]);
  };

  float4 ra[2][NA], rb[2][NB];                      // two tiles on their way, by the parity of their number
  const int full = g.K / S_BK, rest = g.K - full * S_BK;
  auto load = [&](float4 (&va)[NA], float4 (&vb)[NB], int t) {
    load_tile<A_KC, NA, VEC, false>(A, g.lda, m0, t * S_BK, g.M, g.K, va);
    load_tile<B_KC, NB, VEC, false>(B, g.ldb, n0, t * S_BK, g.N, g.K, vb);
  };
  bf16x8 fa[3][TM], fb[3][TN];
  auto get = [&](const char *buf) {
    read_split<BN, TN>(buf + ABYTES, wn, lr, lk, fb);
    read_split<BM, TM>(buf, wm, lr, lk, fa);
  };
  // Tile t is multiplied while tile t + 1 goes from registers through the split into the other buffer; tile t + 2 is on its way and
  // tile t + 3 is requested, each value as soon as the one before it in its registers has been cut.  (Past the last whole tile the last
  // one is loaded again and not used.)  FIRST: the first step of S_FLUSH, which adds the short sums of the steps before it to the long
  // ones and starts new ones.
  auto step = [&](auto first, auto parity, int t) {
    constexpr bool FIRST = decltype(first)::value;
    constexpr int ODD = decltype(parity)::value ? 1 : 0;
    get(smem + ODD * (ABYTES + BBYTES));
    if (FIRST) flush();
    mfma6_tiles<FIRST>(fa, fb, acc);
    char *next = smem + (ODD ^ 1) * (ABYTES + BBYTES);
    const int k0 = min(t + 3, full - 1) * S_BK;
#pragma unroll
    for (int i = 0; i < NA; i++) {
      store_part<A_KC, BM, false>(next, ra[ODD ^ 1][i], i);
      ra[ODD ^ 1][i] = load_part<A_KC, VEC, false>(A, g.lda, m0, k0, g.M, g.K, i);
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
      store_part<B_KC, BN, false>(next + ABYTES, rb[ODD ^ 1][i], i);
      rb[ODD ^ 1][i] = load_part<B_KC, VEC, false>(B, g.ldb, n0, k0, g.N, g.K, i);
    }
    // The fragments of the first two products, then one matrix instruction (32 cycles) and the vector instructions of the split that fit
    // beside it, in turn; the middle parts are read once the lowest ones, whose registers they take, have been multiplied.
    if (TM * TN > 1) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * (TM + TN), 0);
#pragma unroll
      for (int i = 0; i < 6 * TM * TN; i++) {
        if (FIRST && i < TM * TN) __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
        if (i == TM * TN - 1) __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
        if (i & 1) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        if (i % 6 == 5) __builtin_amdgcn_sched_group_barrier(0x020, 4, 0);
      }
    }
    __syncthreads();
  };
  using yes = std::integral_constant<bool, true>;
  using no = std::integral_constant<bool, false>;
  int t = 0;
  if (full > 0) {
    load(ra[0], rb[0], 0);
    load(ra[1], rb[1], min(1, full - 1));
    store_split<A_KC, BM, false>(smem, ra[0]);
    store_split<B_KC, BN, false>(smem + ABYTES, rb[0]);
    load(ra[0], rb[0], min(2, full - 1));
    __syncthreads();
    for (; t + S_FLUSH <= full; t += S_FLUSH) {
      step(yes(), no(), t);
      step(no(), yes(), t + 1);
      step(no(), no(), t + 2);
      step(no(), yes(), t + 3);
    }
    if (t < full) {
      step(yes(), no(), t);
      if (t + 1 < full) step(no(), yes(), t + 1);
      if (t + 2 < full) step(no(), no(), t + 2);
    }
  }
  if (rest > 0) {
    load_tile<A_KC, NA, VEC, true>(A, g.lda, m0, full * S_BK, g.M, g.K, ra[0]);
    load_tile<B_KC, NB, VEC, true>(B, g.ldb, n0, full * S_BK, g.N, g.K, rb[0]);
    store_split<A_KC, BM, true>(smem, ra[0]);
    store_split<B_KC, BN, true>(smem + ABYTES, rb[0]);
    __syncthreads();
    get(smem);
    if (full % S_FLUSH == 0) {
      flush();
      mfma6_tiles<true>(fa, fb, acc);
    } else {
      mfma6_tiles<false>(fa, fb, acc);
    }
    __syncthreads();
  }
  flush();
  bool fine = true;
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) fine = fine && all_finite(sum[i][j]);
  if (__syncthreads_or(!fine)) {
    f32_tile<A_KC, B_KC, BM, BN, VEC>(g, A, B, cbase, m0, n0, vec_c, out_bf16, (float *)smem);
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) finish_tile<PLAIN>(g, cbase, m0 + wm + 32 * i, n0 + wn + 32 * j, sum[i][j], vec_c, out_bf16, smem + wave * 4096);
}

// ================================================================ small products: straight from memory
// A workgroup's WAVES waves share one 32 x 32 tile: wave w contracts the pieces w, w + WAVES, ... of 16 along K, its operands loaded
// from global memory in the layout the matrix instruction wants (lane: row lane%32, the 8 k of half lane/32), four pieces in flight,
// and the partial tiles are added up in LDS in the order of the waves.  No barrier until then.
template <bool KCONTIG>
__device__ __forceinline__ void load_piece(const float *__restrict__ base, int64_t ld, int row, int k, int K, bool vec, float (&v)[8]) {
  const float *p = KCONTIG ? base + (int64_t)row * ld + k : base + (int64_t)k * ld + row;
  const int64_t step = KCONTIG ? 1 : ld;
  if (KCONTIG && vec && k + 8 <= K) {
    const float4 x = reinterpret_cast<const float4 *>(p)[0], y = reinterpret_cast<const float4 *>(p)[1];
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w; v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
  } else if (k + 8 <= K) {
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = p[e * step];
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = k + e < K ? p[e * step] : 0.f;
  }
}
template <bool A_KC, bool B_KC, int WAVES, bool EXACT>
__device__ __forceinline__ void contract_pieces(const GemmArgs &g, const float *A, const float *B, int m0, int n0, bool vec_a, bool vec_b, f32x16 &sum) {
  constexpr int U = 4;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const int ra = min(m0 + lr, g.M - 1), rb = min(n0 + lr, g.N - 1), nc = (g.K + 15) >> 4;
#pragma unroll
  for (int e = 0; e < 16; e++) sum[e] = 0.f;
  for (int c0 = wave; c0 < nc; c0 += WAVES * U) {
    float a[U][8], b[U][8];
    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.f;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = (c0 + u * WAVES) * 16 + 8 * lk;             // a piece past the end loads zeros
      load_piece<A_KC>(A, g.lda, ra, k, g.K, vec_a, a[u]);
      load_piece<B_KC>(B, g.ldb, rb, k, g.K, vec_b, b[u]);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (EXACT) {
#pragma unroll
        for (int e = 0; e < 8; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b[u][e], a[u][e], acc, 0, 0, 0);
      } else {
        bf16x8 fa[3], fb[3];
#pragma unroll
        for (int e = 0; e < 8; e++) { a[u][e] = here(a[u][e]) * SPLIT_UP; b[u][e] = here(b[u][e]) * SPLIT_UP; }
        split8(a[u], fa);
        split8(b[u], fb);
        mfma6(fb, fa, acc);                                     // C^T
      }
    }
#pragma unroll
    for (int e = 0; e < 16; e++) sum[e] = __builtin_fmaf(acc[e], EXACT ? 1.0f : SPLIT_DOWN, sum[e]);      // short sums, added rounded to nearest (S_FLUSH)
  }
}
template <int LAYOUT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_gemm_f32_pieces(GemmArgs g, int vec_a, int vec_b, int vec_c, int out_bf16) {
  constexpr bool A_KC = (LAYOUT != AH_GEMM_TN), B_KC = (LAYOUT == AH_GEMM_NT);
  __shared__ __attribute__((aligned(16))) char smem[WAVES * 4096];
  const float *A = (const float *)g.a + (int64_t)blockIdx.z * g.sa;
  const float *B = (const float *)g.b + (int64_t)blockIdx.z * g.sb;
  const int64_t cbase = (int64_t)blockIdx.z * g.sc;
  int tm, tn;
  tile_of(blockIdx.x, (g.M + 31) / 32, (g.N + 31) / 32, tm, tn);
  const int wave = threadIdx.x >> 6, r = threadIdx.x >> 3, ch = threadIdx.x & 7;
  f32x16 acc;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  auto join = [&]() {
    stage_tile(smem + wave * 4096, acc);
    __syncthreads();
    if (threadIdx.x < 256) {
      s = staged(smem, r, ch);
#pragma unroll
      for (int w = 1; w < WAVES; w++) {
        const float4 v = staged(smem + w * 4096, r, ch);
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
      }
    }
  };
  contract_pieces<A_KC, B_KC, WAVES, false>(g, A, B, tm * 32, tn * 32, vec_a, vec_b, acc);
  join();
  const float z = __builtin_fmaf(s.x, 0.f, __builtin_fmaf(s.y, 0.f, __builtin_fmaf(s.z, 0.f, s.w * 0.f)));      // NaN if one is not finite
  if (__syncthreads_or(!(z == 0.f))) {
    contract_pieces<A_KC, B_KC, WAVES, true>(g, A, B, tm * 32, tn * 32, vec_a, vec_b, acc);
    join();
  }
  if (threadIdx.x < 256) finish4<false>(g, cbase, tm * 32 + r, tn * 32 + 4 * ch, s, vec_c, out_bf16);
}

// The slices of a product added up in their order, and its epilogue: a residual, gelu (both outputs) or gelu's backward.  Memory-bound like the
// plain join (which adds slices only).  A product and an addition of their own became one product, 16384 x 256 x 1024 in two slices
// 73.4 -> 65.3 us, 1024 x 128 x 512 in eight 11.6 -> 9.9, 16384 x 768 x 768 in one piece 135 -> 119.
// gelu as a pass of its own / joined here / in the epilogue of a product that has to stay in one piece for it: 33 x 5120 x 5120 in 16 slices
// 35.5 / 31.9 / 114.6 us, 64 x 4096 x 4096 in four 29.1 / 26.2 / 50.0, 490 x 8192 x 2048 in two 110 / 106 / 118; its backward at the same
// shapes 36.8 / 33.5 / 77.6, 32.0 / 30.0 / 46.7, 113 / 107 / 125.
template <int EPI>
__global__ __launch_bounds__(256) void k_join_epilogue(const float *__restrict__ ws, GemmArgs g, int slices, int64_t n4) {
  const int row4 = g.N / 4;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x) {
    float4 s = reinterpret_cast<const float4 *>(ws)[i];
    for (int k = 1; k < slices; k++) {
      const float4 v = reinterpret_cast<const float4 *>(ws)[k * n4 + i];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    epilogue4<EPI, float>(g, 0, (int)(i / row4), (int)(i % row4) * 4, s.x, s.y, s.z, s.w, true);
  }
}
template <int EPI>
int32_t join_epilogue(const float *ws, const GemmArgs &ga, int slices) {
  const int64_t n4 = (int64_t)ga.M * ga.N / 4;
  ah::launch_kernel(k_join_epilogue<EPI>, dim3((unsigned)(cdiv(n4, 256) < 4096 ? cdiv(n4, 256) : 4096)), dim3(256), 0, ws, ga, slices, n4);
  AH_LAUNCH_CHECK();
  return AH_OK;
}
int32_t join(const float *ws, const GemmArgs &ga, int slices) {
  switch (ga.epi) {
    case AH_EPI_RESIDUAL: return join_epilogue<AH_EPI_RESIDUAL>(ws, ga, slices);
    case AH_EPI_GELU: return join_epilogue<AH_EPI_GELU>(ws, ga, slices);
    case AH_EPI_GELU_BWD: return join_epilogue<AH_EPI_GELU_BWD>(ws, ga, slices);
    default: return ah::splitk_reduce(ws, (float *)ga.c, slices, ga.M, ga.N, ga.ldc, ga.epi == AH_EPI_ACCUM);
  }
}

// ================================================================ dispatch
template <int LAYOUT, int BM, int BN>
int32_t launch_split(const GemmArgs &ga, int batch, int vec_a, int vec_b, int vec_c, int out_bf16) {
  const dim3 grid((unsigned)(cdiv(ga.M, BM) * cdiv(ga.N, BN)), 1, (unsigned)batch);
  note_gemm_kernel("k_gemm_f32_split<%d, %d, %d>", LAYOUT, BM, BN);
  const bool vec = (vec_a || LAYOUT == AH_GEMM_TN) && (vec_b || LAYOUT != AH_GEMM_NT);       // of the operands whose rows run along k
  auto go = [&](auto kfn) { ah::launch_kernel(kfn, grid, dim3(256), 0, ga, vec_c, out_bf16); };
  if (!vec) go(k_gemm_f32_split<LAYOUT, BM, BN, false, false>);
  else if (ga.epi == AH_EPI_NONE && !out_bf16) go(k_gemm_f32_split<LAYOUT, BM, BN, true, true>);
  else go(k_gemm_f32_split<LAYOUT, BM, BN, false, true>);
  AH_LAUNCH_CHECK();
  return AH_OK;
}
template <int LAYOUT, int WAVES>
int32_t launch_pieces(const GemmArgs &ga, int batch, int vec_a, int vec_b, int vec_c, int out_bf16) {
  const dim3 grid((unsigned)(cdiv(ga.M, 32) * cdiv(ga.N, 32)), 1, (unsigned)batch);
  note_gemm_kernel("k_gemm_f32_pieces<%d, %d>", LAYOUT, WAVES);
  ah::launch_kernel((k_gemm_f32_pieces<LAYOUT, WAVES>), grid, dim3(64 * WAVES), 0, ga, vec_a, vec_b, vec_c, out_bf16);
  AH_LAUNCH_CHECK();
  return AH_OK;
}

// bm = 32: 32 x 32 tiles straight from memory, `waves` waves each; otherwise tiles of bm x bm through LDS.  splits: the contraction is cut
// into that many slices, which run as batch entries into a workspace and are then added up in fixed order.
// us: what the choice is expected to take.
struct F32Choice { int bm, waves, splits; double us; };

// The choice is the least of what the candidates are expected to take, in microseconds beyond a launch, from figures measured over 71 shapes
// (1 x 4096 x 1024 to 16384 x 50304 x 768, in the three layouts) on the kernels as they were when a pair of values was cut in 13
// instructions: the tiles have become 2 to 15 % faster since, and the constants are those of then:
//   32 x 32     FIRST, the first round trip; then GROUP per 4 pieces of a wave, and the rate that all of them together reach
//   LDS tiles   a tile takes `step` per 16 of the contraction alone on its CU, and `full` of the CU's time where others fill its gaps
//   slices      another launch, and the workspace written and read
// Against 128 x 128 tiles of v_mfma_f32_32x32x2_f32 (in slices where there were fewer than 256 tiles and K >= 2048), in us:
//   16384 x 3072 x 768 NT 720 -> 436 (128 x 128), 768 x 768 x 16384 TN 329 -> 139 (128 x 128 in 32 slices), 490 x 768 x 768 NT 77 -> 14
//   (64 x 64 in 2 slices), 48 x 768 x 256 NT 26 -> 7 and 512 x 128 x 1024 TN 97 -> 9 (32 x 32).  Operands that are not finite take the
//   fp32 instruction as well: 16384 x 3072 x 768 of NaNs 975 (720 by that instruction's own kernel).
F32Choice choose(const GemmArgs &ga, int layout, int batch, bool may_split, bool long_rows) {
  struct Tile { int bm; double step, full; };
  static constexpr Tile TILES[2] = {{64, 0.26, 0.24}, {128, 1.2, 0.65}};
  static constexpr double FIRST[2] = {0.56, 1.1}, GROUP[2] = {0.74, 0.58}, RATE[3] = {61e6, 50e6, 100e6};      // NN, NT, TN: operations per us
  const double M = ga.M, N = ga.N, K = ga.K;
  // a launch has fewer than 2^32 threads: a row of more than 2^30 columns leaves only the widest tiles
  auto fits = [&](int bm, int threads) { return cdiv(ga.M, bm) * cdiv(ga.N, bm) * threads < (1ll << 32); };
  F32Choice best{32, 8, 1, 1e300};
  for (int w = 0; w < 2; w++) {
    const int waves = 4 << w;
    if (!fits(32, 64 * waves)) continue;
    double t = FIRST[w] + GROUP[w] * (double)cdiv(cdiv(ga.K, 16), waves * 4) +
               (double)(cdiv(ga.M, 32) * cdiv(ga.N, 32) * batch) * 2048.0 * K / RATE[layout] * (w == 0 ? 1.0 : 1.6);
    if (t < best.us) best = F32Choice{32, waves, 1, t};
  }
  if (long_rows) return best;
  for (const Tile &q : TILES)
    for (int s = 1; fits(q.bm, 256) && s <= (may_split ? 32 : 1); s *= 2) {
      if (s > 1 && (K / s < 64 || s * M * N > (1 << 27))) break;
      const double per_cu = (double)(cdiv(ga.M, q.bm) * cdiv(ga.N, q.bm) * batch * s) / num_cus();
      const double b = per_cu < 4 ? ceil(per_cu) : per_cu + 0.5, alone = q.step * (layout == AH_GEMM_TN ? 1.1 : 1.0);
      const double t = K / s / 16 * (b * q.full > alone ? b * q.full : alone) + (s > 1 ? 1.8 + (s + 1) * M * N * 4 / 2.8e6 : 0.0);
      if (t < best.us) best = F32Choice{q.bm, 0, s, t};
    }
  return best;
}

template <int LAYOUT>
int32_t launch_choice(const F32Choice &c, const GemmArgs &ga, int batch, int vec_a, int vec_b, int vec_c, int out_bf16) {
  if (c.bm == 32) {
    return c.waves == 4 ? launch_pieces<LAYOUT, 4>(ga, batch, vec_a, vec_b, vec_c, out_bf16)
                        : launch_pieces<LAYOUT, 8>(ga, batch, vec_a, vec_b, vec_c, out_bf16);
  }
  if (c.bm == 64) return launch_split<LAYOUT, 64, 64>(ga, batch, vec_a, vec_b, vec_c, out_bf16);
  return launch_split<LAYOUT, 128, 128>(ga, batch, vec_a, vec_b, vec_c, out_bf16);
}

// Where the memory for the slices is refused, the product runs without any.
int32_t run_choice(const F32Choice &c, const GemmArgs &ga, int layout, int batch, int out_dtype, int vec_a, int vec_b, int vec_c, bool long_rows) {
  const int ob = out_dtype == AH_BF16;
  auto go = [&](const GemmArgs &g, int nb, int vc) -> int32_t {
    switch (layout) {
      case AH_GEMM_NN: return launch_choice<AH_GEMM_NN>(c, g, nb, vec_a, vec_b, vc, ob);
      case AH_GEMM_NT: return launch_choice<AH_GEMM_NT>(c, g, nb, vec_a, vec_b, vc, ob);
      default: return launch_choice<AH_GEMM_TN>(c, g, nb, vec_a, vec_b, vc, ob);
    }
  };
  const int64_t slice = (cdiv(ga.K, c.splits) + 15) & ~15ll;          // whole steps of 16, so that every slice is aligned as the whole is
  const int slices = c.splits > 1 ? (int)cdiv(ga.K, slice) : 1;
  if (slices <= 1) {
    const int32_t rc = go(ga, batch, vec_c);
    note_gemm_split(1);
    return rc;
  }
  ah_ptr ws = 0;
  int32_t rc = ah_alloc((uint64_t)slices * ga.M * ga.N * 4, &ws);
  if (rc == AH_ERR_OOM) return run_choice(choose(ga, layout, batch, false, long_rows), ga, layout, batch, out_dtype, vec_a, vec_b, vec_c, long_rows);
  if (rc) return rc;
  GemmArgs gs = ga;
  gs.ksplit = (int)slice; gs.nsplit = slices;
  gs.sa = layout == AH_GEMM_TN ? slice * ga.lda : slice;
  gs.sb = layout == AH_GEMM_NT ? slice : slice * ga.ldb;
  gs.c = dp<void>(ws); gs.ldc = ga.N; gs.sc = (int64_t)ga.M * ga.N; gs.epi = AH_EPI_NONE;
  rc = go(gs, slices, 1);
  if (rc == AH_OK) rc = join(dp<const float>(ws), ga, slices);
  note_gemm_split(slices);
  const int32_t rf = ah_free(ws);      // stream-ordered: reusable only by later work
  return rc ? rc : rf;
}

}  // namespace

namespace ah {
// ga.nsplit: 0 keeps a product in one piece
int32_t gemm_f32(const GemmArgs &ga, int layout, int batch, int out_dtype, int vec_a, int vec_b, int vec_c) {
  const bool joins = ga.epi == AH_EPI_NONE || ga.epi == AH_EPI_ACCUM || ga.epi == AH_EPI_RESIDUAL || ga.epi == AH_EPI_GELU || ga.epi == AH_EPI_GELU_BWD;
  const bool may_split = ga.nsplit > 0 && batch == 1 && out_dtype == AH_F32 && joins && ga.N % 4 == 0 && vec_c;
  // the tile loaders' offsets within a tile are 32 bits: its rows, 128 at most, span less than 4 GiB
  auto spans = [](int rows, int64_t ld) { return ((rows < 128 ? rows : 128) - 1) * ld + 16 >= (1ll << 30); };
  const bool long_rows = (layout != AH_GEMM_TN && spans(ga.M, ga.lda)) || (layout == AH_GEMM_NT && spans(ga.N, ga.ldb));
  F32Choice c = choose(ga, layout, batch, may_split, long_rows);
  // With gelu or its backward one piece is one launch and slices are two and a workspace, where the plain product's slices are what its join is
  // compared with.  So slices have to be expected to gain something: 2.5 us on tiles through LDS, 6 on 32 x 32 pieces, whose estimate is
  // that much too high beside a join.  Measured in graphs, slices / one piece, forward and backward: tiles that gain 0 to 2.1 us by the
  // estimate 27.7 / 28.4 and 27.5 / 30.7 (274 x 3456 x 864) to 63.6 / 60.5 and 62.0 / 63.0 (912 x 4096 x 1024), and a second launch
  // is some 4 us of the host, which is what bounds a pass of a small model; from 2.5 us on 15.8 / 20.9 and 17.0 / 23.1 (108 x 3584 x
  // 896), 42.3 / 45.3 and 44.5 / 50.8 (256 x 6144 x 1536).  Pieces that gain 0 to 4.5 us 9.8 / 10.1 and 10.3 / 8.1 (88 x 2048 x 512),
  // 13.2 / 12.7 and 14.1 / 10.6 (65 x 2688 x 672), backward 14.1 / 13.3 (64 x 4096 x 1024); from 6 us on 13.5 / 17.4 (its forward pass),
  // 18.1 / 28.8 and 20.0 / 23.5 (128 x 2048 x 2048).
  if (c.splits > 1 && (ga.epi == AH_EPI_GELU || ga.epi == AH_EPI_GELU_BWD)) {
    const F32Choice one = choose(ga, layout, batch, false, long_rows);
    if (one.us - c.us < (one.bm == 32 ? 6.0 : 2.5)) c = one;
  }
  return run_choice(c, ga, layout, batch, out_dtype, vec_a, vec_b, vec_c, long_rows);
}
}  // namespace ah
