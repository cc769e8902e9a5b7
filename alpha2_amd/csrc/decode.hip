// One token through the model, from the keys and values that earlier tokens left (packages/train/src/sample.ts:36-198 runs the whole
// context again for each new token; a causal row depends on the rows before it through their keys and values only).
//
// A single row makes every product a matrix times a vector: nothing is used twice, so there is no tile to share and the bound is the
// weights read once (4 bytes for 2 operations) - where a launch is long enough to feel it.  At the sizes sampled in earnest (256 to
// 1024 wide) a matrix is 0.3 to 12 MB, a microsecond or two of the chip, and what a token takes is the chain of dependent launches.
// So the launches are few, one for the whole token of small models (k_decode_chain) and otherwise five a layer, each does the small work in front of its product itself, and each asks for its weights before
// anything it has to wait for:
//   k_decode_rows<NORM>  LayerNorm (the first one of all adds the two embeddings) + q, k, v into the row of the cache; + fc1 and its
//                        activation (gate and up together); + the head.  Every wave normalises the row again, in registers.
//   k_decode_attention   keys in slices of at least 64, one workgroup to a slice and head
//   k_decode_rows<JOIN>  joins the slices (softmax weights of the slices' maxima) in LDS + wo + the residual stream
//   k_decode_long        fc2 + the residual stream: long rows, few of them, so four waves to a row
// 64 tokens from a 6 x 256 model 56.0 -> 11.5 ms in launches and 9.0 in one launch a token, 24 tokens behind a prompt of 480 from the GPT-2-small shape 59.9 -> 11.4 (each with
// the pass over the finished sequence that follows).  A launch takes 2.9 to 5.7 us there and the next one starts about 1 us later.
#include "common.h"
#include <algorithm>
#include <atomic>
#include <cmath>

using namespace ah;

namespace {

constexpr int MAX_SLICES = 16, MIN_SLICE = 64;
constexpr int MAX_WIDTH = 4096;                 // the row in registers: 16 float4 a lane

struct DecodeRows {
  const float *x;                               // NORM: the row to normalise; JOIN: the slices' sums [slices][K]
  const float *gain, *bias;                     // NORM
  const float *tok, *pos;                       // NORM: not null: the row is tok + pos, and `stream` takes it
  const float2 *top;                            // JOIN: (maximum, sum of exponentials) [slices][heads]
  const float *w, *w_up;                        // [N][K]; DUAL: gate and up
  float *stream, *out;                          // out: null: the results are added to `stream`
  const float *coef[5];                         // activation: sum over the bases of `mask` (bit 0 silu, 1 relu, 2 gelu, 3 identity,
  int mask;                                     // 4 square) of coef[n] (null: 1) times basis; 0: none
  int N, K, slices, heads;
  float eps;
};

__device__ __forceinline__ float silu(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float activate(const DecodeRows &a, int n, float x) {
  if (a.mask == 0) return x;
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < 5; k++) {
    if (!(a.mask >> k & 1)) continue;
    const float v = k == 0 ? silu(x) : k == 1 ? (x > 0.f ? x : 0.f) : k == 2 ? gelu_f(x) : k == 3 ? x : x * x;
    s += a.coef[k] ? a.coef[k][n] * v : v;
  }
  return s;
}
__device__ __forceinline__ float4 ldq(const float *p, int j) { return reinterpret_cast<const float4 *>(p)[j]; }
__device__ __forceinline__ float dot4(float4 a, float4 b, float s) {
  return __builtin_fmaf(a.w, b.w, __builtin_fmaf(a.z, b.z, __builtin_fmaf(a.y, b.y, __builtin_fmaf(a.x, b.x, s))));
}

// what sums about the maximum m count for beside those about `most`; -inf: no key
__device__ __forceinline__ float slice_weight(float m, float most) { return m == -INFINITY ? 0.f : expf(m - most); }

enum { NORM = 0, JOIN = 1 };
// A wave computes R neighbouring results (DUAL: R of the gate and R of the up matrix).  NV: float4 per lane of a row, K <= 256 NV.
template <int PRO, int NV, int R, bool DUAL>
__global__ __launch_bounds__(256) void k_decode_rows(DecodeRows a) {
  constexpr int ROWS = DUAL ? 2 * R : R;
  __shared__ __attribute__((aligned(16))) float joined[PRO == JOIN ? 256 * NV : 4];
  __shared__ float weights[PRO == JOIN ? MAX_SLICES * 32 * NV : 4], sums[PRO == JOIN ? 32 * NV : 4];      // heads of 8 features at least
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nv = a.K >> 2, n0 = (blockIdx.x * 4 + wave) * R;
  float4 w[ROWS][NV], x[NV];
#pragma unroll
  for (int r = 0; r < ROWS; r++) {
    const float *row = (DUAL && r >= R ? a.w_up : a.w) + (int64_t)min(n0 + r % R, a.N - 1) * a.K;      // past the end: the last row, not stored
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const int j = lane + 64 * i;
      w[r][i] = j < nv ? ldq(row, j) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  if (PRO == NORM) {
    float4 g[NV], b[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const int j = lane + 64 * i;
      const bool in = j < nv;
      x[i] = g[i] = b[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (in) {
        g[i] = ldq(a.gain, j);
        b[i] = ldq(a.bias, j);
        x[i] = ldq(a.tok ? a.tok : a.x, j);
        if (a.tok) {
          const float4 p = ldq(a.pos, j);
          x[i].x += p.x; x[i].y += p.y; x[i].z += p.z; x[i].w += p.w;
          if (blockIdx.x == 0 && wave == 0) reinterpret_cast<float4 *>(a.stream)[j] = x[i];
        }
      }
    }
    // two passes over the registers, as k_layernorm
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++) s += (x[i].x + x[i].y) + (x[i].z + x[i].w);
    const float inv = 1.0f / (float)a.K, mean = wave_sum(s) * inv;
#pragma unroll
    for (int i = 0; i < NV; i++)
      if (lane + 64 * i < nv) {
        const float c = x[i].x - mean, d = x[i].y - mean, e = x[i].z - mean, f = x[i].w - mean;
        q += (c * c + d * d) + (e * e + f * f);
      }
    const float rstd = 1.0f / sqrtf(wave_sum(q) * inv + a.eps);
#pragma unroll
    for (int i = 0; i < NV; i++)
      if (lane + 64 * i < nv)
        x[i] = make_float4((x[i].x - mean) * rstd * g[i].x + b[i].x, (x[i].y - mean) * rstd * g[i].y + b[i].y,
                           (x[i].z - mean) * rstd * g[i].z + b[i].z, (x[i].w - mean) * rstd * g[i].w + b[i].w);
  } else {
    // A thread to a head makes the slices' weights (eight slices asked for at once); meanwhile the slices' sums are on their way, eight at a time.  With
    // the weights made again for every feature this launch took 6.5 us at 768 wide with 8 slices, now 5.2.
    const int head_size = a.K / a.heads;
    constexpr bool AHEAD = NV <= 4;
    float y[AHEAD ? NV : 1][8];
    auto load = [&](int i, int s0, float (&to)[8]) {
      const int k = min(threadIdx.x + 256 * i, a.K - 1);
#pragma unroll
      for (int u = 0; u < 8; u++) to[u] = a.x[(int64_t)min(s0 + u, a.slices - 1) * a.K + k];
    };
    if (AHEAD) {
#pragma unroll
      for (int i = 0; i < NV; i++) load(i, 0, y[AHEAD ? i : 0]);
    }
    for (int h = threadIdx.x; h < a.heads; h += 256) {
      float2 t[MAX_SLICES];
      float top = -INFINITY, sum = 0.f;
#pragma unroll
      for (int s = 0; s < MAX_SLICES; s++) {
        if (s >= 8 && a.slices <= 8) { t[s] = make_float2(-INFINITY, 0.f); continue; }
        t[s] = a.top[min(s, a.slices - 1) * a.heads + h];
        if (s >= a.slices) t[s] = make_float2(-INFINITY, 0.f);
        top = fmaxf(top, t[s].x);
      }
#pragma unroll
      for (int s = 0; s < MAX_SLICES; s++) {
        if (s >= 8 && a.slices <= 8) continue;
        const float c = slice_weight(t[s].x, top);
        sum = __builtin_fmaf(c, t[s].y, sum);
        weights[s * 32 * NV + h] = c;
      }
      sums[h] = sum;
    }
    __syncthreads();
#pragma unroll(AHEAD ? NV : 1)
    for (int i = 0; i < NV; i++) {
      const int k = min(threadIdx.x + 256 * i, a.K - 1), h = k / head_size;
      float v = 0.f;
      for (int s0 = 0; s0 < a.slices; s0 += 8) {
        float z[8];
        if (AHEAD && s0 == 0) {
#pragma unroll
          for (int u = 0; u < 8; u++) z[u] = y[AHEAD ? i : 0][u];
        } else {
          load(i, s0, z);
        }
#pragma unroll
        for (int u = 0; u < 8; u++) v = s0 + u < a.slices ? __builtin_fmaf(weights[(s0 + u) * 32 * NV + h], z[u], v) : v;
      }
      joined[k] = v / sums[h];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const int j = lane + 64 * i;
      x[i] = j < nv ? ldq(joined, j) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  float s[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; r++) {
    s[r] = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++) s[r] = dot4(w[r][i], x[i], s[r]);
  }
#pragma unroll
  for (int r = 0; r < ROWS; r++) s[r] = wave_sum(s[r]);
#pragma unroll
  for (int r = 0; r < R; r++)
    if (lane == r && n0 + r < a.N) {
      const float v = DUAL ? silu(s[r]) * s[(R + r) % ROWS] : activate(a, n0 + r, s[r]);
      if (a.out) a.out[n0 + r] = v;
      else a.stream[n0 + r] += v;
    }
}

// stream[n] += row n of w times x, a workgroup to a row
__global__ __launch_bounds__(256) void k_decode_long(const float *__restrict__ w, const float *__restrict__ x, float *__restrict__ stream, int K) {
  __shared__ float part[4];
  const int nv = K >> 2;
  const float *row = w + (int64_t)blockIdx.x * K;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = threadIdx.x; j0 < nv; j0 += 1024) {
    float4 a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = j0 + 256 * u;
      a[u] = j < nv ? ldq(row, j) : make_float4(0.f, 0.f, 0.f, 0.f);
      b[u] = j < nv ? ldq(x, j) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) s[u] = dot4(a[u], b[u], s[u]);
  }
  const float t = wave_sum((s[0] + s[1]) + (s[2] + s[3]));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) stream[blockIdx.x] += (part[0] + part[1]) + (part[2] + part[3]);
}

// The newest row's query against the keys of one slice, for one head.  G lanes hold a head's features, four each, so a workgroup takes
// 256 / G keys at a time, four of them on their way, and the waves are joined at the end.  Every lane of a group has the group's scores; each takes tanh and
// exp of one (of all, one after the other with a running maximum to a group: 12 heads x 64 behind 500 rows 5.7 -> 4.0 us).
// qkv: the layer's rows of [q | k | v]; sums: [slices][width], not yet divided; top: [slices][heads].
struct DecodeAttention {
  const float *qkv;
  float *sums;
  float2 *top;
  int n, slice, width, head_size;
  float scale, cap;
};
template <int G>
__global__ __launch_bounds__(256) void k_decode_attention(DecodeAttention a) {
  constexpr int KEYS = 256 / G, U = 4;
  __shared__ float all_m[4], all_l[4];
  __shared__ __attribute__((aligned(16))) float all_o[4][4 * G];
  const int h = blockIdx.y, first = blockIdx.x * a.slice, count = min(a.slice, a.n - first);
  const int f = threadIdx.x % G, key = threadIdx.x / G, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bool in = 4 * f < a.head_size;
  const int64_t pitch = 3 * (int64_t)a.width;
  const float *at = a.qkv + h * a.head_size + 4 * (in ? f : 0);
  const float4 none = make_float4(0.f, 0.f, 0.f, 0.f);
  const float4 q = in ? ldq(at + (a.n - 1) * pitch, 0) : none;
  const float *ks = at + first * pitch + a.width;
  float m = -INFINITY, l = 0.f;
  float4 o = none;
  for (int j0 = 0; j0 < count; j0 += KEYS * U) {
    float4 k[U], v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float *p = ks + min(j0 + key + u * KEYS, count - 1) * pitch;
      k[u] = ldq(p, 0);
      v[u] = ldq(p + a.width, 0);
    }
    // the U scores of a group of lanes, one of them to a lane for what tanh and exp take, and one maximum to a wave
    float mine = 0.f;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float s = near_sum<G>(in ? dot4(q, k[u], 0.f) : 0.f);
      mine = (f & (U - 1)) == u ? s : mine;
    }
    mine *= a.scale;
    if (a.cap > 0.f) mine = a.cap * tanhf(mine / a.cap);
    if (j0 + key + (f & (U - 1)) * KEYS >= count) mine = -INFINITY;
    const float most = fmaxf(m, wave_max(mine)), old = slice_weight(m, most), p = f < U ? slice_weight(mine, most) : 0.f;
    l = __builtin_fmaf(l, old, wave_sum(p));
    o.x *= old; o.y *= old; o.z *= old; o.w *= old;
    m = most;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float pu = __shfl(p, (lane & ~(G - 1)) + u, 64);
      o.x = __builtin_fmaf(pu, v[u].x, o.x); o.y = __builtin_fmaf(pu, v[u].y, o.y);
      o.z = __builtin_fmaf(pu, v[u].z, o.z); o.w = __builtin_fmaf(pu, v[u].w, o.w);
    }
  }
  // the groups of a wave, then the waves
  auto far = [&](auto step) { o.x = step(o.x); o.y = step(o.y); o.z = step(o.z); o.w = step(o.w); };
  if (G < 16) far([](float v) { return add_lane<8>(v); });
  if (G < 32) far([](float v) { return add_lane<16>(v); });
  far([](float v) { return add_lane<32>(v); });
  if (lane < G) {
    reinterpret_cast<float4 *>(all_o[wave])[lane] = o;
    if (lane == 0) { all_m[wave] = m; all_l[wave] = l; }
  }
  __syncthreads();
  const float most = fmaxf(fmaxf(all_m[0], all_m[1]), fmaxf(all_m[2], all_m[3]));
  float c[4], sum = 0.f;
#pragma unroll
  for (int w = 0; w < 4; w++) { c[w] = slice_weight(all_m[w], most); sum = __builtin_fmaf(c[w], all_l[w], sum); }
  for (int d = threadIdx.x; d < a.head_size; d += 256) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) v = __builtin_fmaf(c[w], all_o[w][d], v);
    a.sums[(int64_t)blockIdx.x * a.width + h * a.head_size + d] = v;
  }
  if (threadIdx.x == 0) a.top[blockIdx.x * gridDim.y + h] = make_float2(most, sum);
}

// ================================================================ a token in one launch
// The five launches of a layer cost 3 to 6 us each and 1 us between them, whatever they compute.  k_decode_chain runs all of them, and the head,
// as phases of one launch of at most a workgroup to a CU: what a phase hands to the next is written as 64-bit words of a value and a tag, and
// who needs it reads the words until they bear the tag of this layer of this launch.  A word is written and read whole (relaxed atomics of
// device scope), so the tag says that the value beside it is the new one: no flag, no fence, no barrier over the grid, one trip
// through memory from a phase to the next.
//   waves 4 .. 7 wait for the words of the next phase, normalise or join them and leave them in LDS;
//   waves 0 .. 3 meanwhile have the rows of the next matrices (and the keys and values of this workgroup's slice) on their way into registers:
//   the two are different waves because a wave's loads come back in order.
// A buffer is written again a layer later.  Whoever writes it then has read all results of the phase before, which stand on those of all
// phases since the earlier use, and those were computed after their inputs had been read: nobody reads the old words any more.
// All workgroups have to be on the chip at once, which the grid's size allows but nothing guarantees while other processes use the GPU.
// So every wait ends: after SPIN_TICKS, or as soon as another workgroup has given up, a workgroup leaves `chain_gave_up` and ends, and the launch
// behind it computes the token again (and otherwise ends at once).  That one is a single workgroup: its waits are for words that its own waves write, which
// are on the chip when it is, so no clock ends them - time in which the queue is switched off the chip does not count - but a number of tries
// does, that no healthy wait comes near.  Its logits are NaN until it has computed them, and `chain_again` counts it (ah_decode_stats).  The tokens
// behind it take one launch again: sums are cut elsewhere in the launches of a layer, and what a program computes does not depend on who else uses the GPU.
// What bounds it is that chain of trips, 1.3 us at least and 2 to 3 as polled, five a layer, and between them the one wave that has the next step
// (350 instructions in a row are 1 us).  A token, its logits read and chosen from, in launches (whose host work differs that much between processes) and in
// one: 2 x 64 behind 17 rows 64 to 110 / 56 us, 4 x 128 89 to 149 / 86, 32 x 128 behind 100 486 to 608 / 456, 6 x 256 116 to 175 / 121, 8 x 384 153 to
// 198 / 175, behind 200 195 to 253 / 221, 8 x 512 behind 17 163 to 213 / 185.  The kernel alone: 6 x 256 96 us, 16 a layer.  All rows ahead have to be asked for unconditionally: behind branches the
// compiler waits for the newest of them before the oldest (attention 2.3 -> 1.9 us).
constexpr int CHAIN_LAYERS = 32, CHAIN_NV = 2, CHAIN_UNITS = 4;      // at most: layers; 256 NV wide, ffn 1024 NV; keys a lane holds
constexpr int CHAIN_WIDTH = 256 * CHAIN_NV, CHAIN_FFN = 1024 * CHAIN_NV, CHAIN_TOPS = MAX_SLICES * (CHAIN_WIDTH / 8) * 2;      // heads of 8 features at least
constexpr int64_t SPIN_TICKS = 1000000;                              // of 10 ns; computing again takes 0.7 ms (4 x 128) to 9.6 (12 x 512)
constexpr int RESCUE_TRIES = 1 << 24;                                // 10 s and more at a microsecond a try
enum { WORD_QKV = 0, WORD_SUMS = WORD_QKV + 3 * CHAIN_WIDTH, WORD_TOPS = WORD_SUMS + MAX_SLICES * CHAIN_WIDTH, WORD_MID = WORD_TOPS + CHAIN_TOPS,
       WORD_HID = WORD_MID + CHAIN_WIDTH, WORD_STREAM = WORD_HID + CHAIN_FFN, WORDS = WORD_STREAM + CHAIN_WIDTH };
__device__ uint64_t chain_words[WORDS];
__device__ uint32_t chain_gave_up;              // the first tag of the launch that did
__device__ uint64_t chain_again;                // tokens computed again

struct DecodeChain {
  AhDecodeLayer layer[CHAIN_LAYERS];
  ah_ptr lnf_w, lnf_b;
  const float *tok, *pos, *head;
  float *kv, *logits;
  int vocab, width, heads, head_size, ffn, layers, mask, n, slices, slice, lanes;      // lanes: of a head's features, four each, a power of two
  int64_t layer_stride;                         // of kv
  int64_t ticks;                                // a wait's end; in the launch that computes a token again it is `tries`
  int32_t tries;
  float scale, cap, eps;
  uint32_t tag;                                 // layer i's words bear tag + i
  uint32_t rescue;                              // 0, or the first tag of the launch that this one computes again if it gave up
};
static_assert(sizeof(DecodeChain) <= 4096, "kernel arguments");

__device__ __forceinline__ void put(int at, uint32_t tag, float v) {
  __hip_atomic_store(chain_words + at, (uint64_t)tag << 32 | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t peek(int at) { return __hip_atomic_load(chain_words + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// The words index(i), i < N, once all of them (of all lanes) bear the tag; false: given up
template <int N, class Index>
__device__ __forceinline__ bool take(const DecodeChain &a, uint32_t tag, Index index, float (&v)[N]) {
  int64_t since = 0;
  for (int tries = 1;; tries++) {
    uint64_t w[N];
#pragma unroll
    for (int i = 0; i < N; i++) w[i] = peek(index(i));
    uint32_t other = 0;
#pragma unroll
    for (int i = 0; i < N; i++) { other |= (uint32_t)(w[i] >> 32) ^ tag; v[i] = __uint_as_float((uint32_t)w[i]); }
    if (__all(other == 0)) return true;
    if (a.rescue) {
      if (tries >= a.tries) return false;
    } else if ((tries & 63) == 0 || a.ticks < 0) {
      const int64_t now = wall_clock64();
      if (since == 0) since = now;
      if (now - since > a.ticks || __hip_atomic_load(&chain_gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.tag) {
        __hip_atomic_store(&chain_gave_up, a.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
    }
  }
}

// the sum over the lanes of a group of g (8 to 64), in each of them
__device__ __forceinline__ float group_sum(float v, int g) {
  v = near_sum<8>(v);
  if (g >= 16) v = add_lane<8>(v);
  if (g >= 32) v = add_lane<16>(v);
  return g >= 64 ? add_lane<32>(v) : v;
}

template <int NV, bool DUAL>
__global__ __launch_bounds__(512, 2) void k_decode_chain(DecodeChain a) {
  constexpr int PAIRS = DUAL ? (NV + 1) / 2 : 0, RA = DUAL ? 2 * PAIRS : NV, NF = 4 * NV, U = CHAIN_UNITS, E = 4 * NV;
  __shared__ __attribute__((aligned(16))) float xn[256 * NV], joined[256 * NV], hid[1024 * NV];
  __shared__ float stream[256 * NV], mid[256 * NV];
  __shared__ __attribute__((aligned(16))) float fresh[3][128];         // the new row's q, k, v of a head
  __shared__ __attribute__((aligned(16))) float part_o[4][128];
  __shared__ float part_m[4], part_l[4], tops[CHAIN_TOPS];
  __shared__ int quit[2];
  if (a.rescue && __hip_atomic_load(&chain_gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != a.rescue) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, C = a.width, F = a.ffn, nv = C >> 2, nf = F >> 2;
  const int G = gridDim.x, W = 4 * G, gw = blockIdx.x * 4 + wave;      // row gw + r W of a matrix is this wave's
  const int units = a.slices * a.heads;
  const bool in_c = blockIdx.x * 4 < (unsigned)C, in_qkv = blockIdx.x * 4 < (unsigned)(3 * C), in_f = blockIdx.x * 4 < (unsigned)F;
  if (threadIdx.x < 2) quit[threadIdx.x] = 0;
  if (a.rescue) {
    for (int i = threadIdx.x; i < a.vocab; i += 512) a.logits[i] = __builtin_nanf("");
    if (threadIdx.x == 0) __hip_atomic_fetch_add(&chain_again, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  // A barrier behind which all waves see the same: has one given up before it?  Two words in turns, since a wave may have given up on the next phase
  // before another has read what the last one left.
  int turn = 0;
  auto meet = [&]() {
    __syncthreads();
    turn ^= 1;
    return quit[turn ^ 1] != 0;
  };

  auto at = [](ah_ptr p) { return reinterpret_cast<const float *>(static_cast<uintptr_t>(p)); };
  // The two kinds of waves run loops of their own, so that neither's registers are kept through the other's code; both come to the same barriers.
  if (wave >= 4) {
    const int ct = threadIdx.x - 256;
    float gain[E], bias[E];
    auto load_norm = [&](ah_ptr g, ah_ptr b) {
#pragma unroll
      for (int i = 0; i < E; i++) { const int k = lane + 64 * i; gain[i] = k < C ? at(g)[k] : 0.f; bias[i] = k < C ? at(b)[k] : 0.f; }
    };
    // x: elements lane + 64 i of the row, which `raw` takes as they are and xn normalised, in two passes over the registers
    auto norm = [&](const float (&x)[E], float *raw) {
      float s = 0.f, q = 0.f;
#pragma unroll
      for (int i = 0; i < E; i++) s += lane + 64 * i < C ? x[i] : 0.f;
      const float inv = 1.0f / (float)C, mean = wave_sum(s) * inv;
#pragma unroll
      for (int i = 0; i < E; i++) { const float c = x[i] - mean; q += lane + 64 * i < C ? c * c : 0.f; }
      const float rstd = 1.0f / sqrtf(wave_sum(q) * inv + a.eps);
#pragma unroll
      for (int i = 0; i < E; i++) {
        const int k = lane + 64 * i;
        if (k < C) { raw[k] = x[i]; xn[k] = (x[i] - mean) * rstd * gain[i] + bias[i]; }
      }
    };
    auto take_row = [&](int words, uint32_t tag, float (&x)[E]) {
      if (!take<E>(a, tag, [&](int i) { return words + min(lane + 64 * i, C - 1); }, x)) quit[turn] = 1;
    };
    int head2[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) head2[i] = min(ct + 256 * i, C - 1) / a.head_size * 2;
    if (wave == 4) load_norm(a.layer[0].ln1_w, a.layer[0].ln1_b);
#pragma unroll 1
    for (int l = 0; l < a.layers; l++) {
      const uint32_t tag = a.tag + l;
      if (in_qkv) {
        if (wave == 4) {
          float x[E];
          if (!in_f && !in_c) load_norm(a.layer[l].ln1_w, a.layer[l].ln1_b);
          if (l == 0) {
#pragma unroll
            for (int i = 0; i < E; i++) { const int k = lane + 64 * i; x[i] = k < C ? a.tok[k] + a.pos[k] : 0.f; }
          } else {
            take_row(WORD_STREAM, tag - 1, x);
          }
          norm(x, stream);
          load_norm(a.layer[l].ln2_w, a.layer[l].ln2_b);
        }
        if (meet()) return;
      }
      for (int unit = blockIdx.x; unit < units; unit += G) {
        if (ct < 128) {
          float x[3];
          const int from = WORD_QKV + unit % a.heads * a.head_size + min(ct, a.head_size - 1);
          if (!take<3>(a, tag, [&](int i) { return from + i * C; }, x)) quit[turn] = 1;
#pragma unroll
          for (int i = 0; i < 3; i++) fresh[i][ct] = x[i];
        }
        if (meet()) return;
        __syncthreads();
      }
      if (in_c) {
        // the slices' maxima and sums go through LDS; then the slices are joined, S at a time
        constexpr int S = 4;
        const int ntops = units * 2;
        float x[NV * S + 1];
        auto sums = [&](int s0, int e) { return WORD_SUMS + min(s0 + e % S, a.slices - 1) * C + min(ct + 256 * (e / S), C - 1); };
        if (!take<NV * S + 1>(a, tag, [&](int e) { return e == 0 ? WORD_TOPS + min(ct, ntops - 1) : sums(0, e - 1); }, x)) quit[turn] = 1;
        if (ct < ntops) tops[ct] = x[0];
        for (int t = ct + 256; t - ct < ntops; t += 256) {
          float y[1];
          if (!take<1>(a, tag, [&](int) { return WORD_TOPS + min(t, ntops - 1); }, y)) quit[turn] = 1;
          if (t < ntops) tops[t] = y[0];
        }
        if (meet()) return;
        float most[NV], sum[NV], v[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) { most[i] = -INFINITY; sum[i] = v[i] = 0.f; }
        for (int s0 = 0; s0 < a.slices; s0 += S) {
          float y[NV * S];
          if (s0 > 0 && !take<NV * S>(a, tag, [&](int e) { return sums(s0, e); }, y)) { quit[turn] = 1; break; }
#pragma unroll
          for (int i = 0; i < NV; i++) {
            const float *top = tops + head2[i];
            float now = most[i];
#pragma unroll
            for (int s = 0; s < S; s++) if (s0 + s < a.slices) now = fmaxf(now, top[(s0 + s) * a.heads * 2]);
            const float old = slice_weight(most[i], now);
            sum[i] *= old;
            v[i] *= old;
            most[i] = now;
#pragma unroll
            for (int s = 0; s < S; s++)
              if (s0 + s < a.slices) {
                const float *t = top + (s0 + s) * a.heads * 2, c = slice_weight(t[0], now);
                sum[i] = __builtin_fmaf(c, t[1], sum[i]);
                v[i] = __builtin_fmaf(c, s0 == 0 ? x[i * S + s + 1] : y[i * S + s], v[i]);
              }
          }
        }
#pragma unroll
        for (int i = 0; i < NV; i++) if (ct + 256 * i < C) joined[ct + 256 * i] = v[i] / sum[i];
        if (meet()) return;
      }
      if (in_f || in_c) {
        if (wave == 4) {
          float x[E];
          if (!in_qkv) load_norm(a.layer[l].ln2_w, a.layer[l].ln2_b);
          take_row(WORD_MID, tag, x);
          norm(x, mid);
          const bool last = l + 1 == a.layers;
          load_norm(last ? a.lnf_w : a.layer[l + 1].ln1_w, last ? a.lnf_b : a.layer[l + 1].ln1_b);
        }
        if (meet()) return;
      }
      if (in_c) {
        float x[E];
        if (!take<E>(a, tag, [&](int i) { return WORD_HID + min(ct + 256 * i, F - 1); }, x)) quit[turn] = 1;
#pragma unroll
        for (int i = 0; i < E; i++) if (ct + 256 * i < F) hid[ct + 256 * i] = x[i];
        if (meet()) return;
      }
    }
    if (wave == 4) {
      float x[E];
      if (!in_f && !in_c) load_norm(a.lnf_w, a.lnf_b);
      take_row(WORD_STREAM, a.tag + a.layers - 1, x);
      norm(x, stream);
    }
    meet();
    return;
  }

  float4 wa[RA][NV], wo[NV], w2[NF], kk[U], vv[U];
  auto row_of = [&](float4 (&w)[NV], const float *m, int n, int N) {
#pragma unroll
    for (int i = 0; i < NV; i++) {
      w[i] = ldq(m + (int64_t)min(n, N - 1) * C, min(lane + 64 * i, nv - 1));
    }
  };
  auto long_row = [&](const float *m, int n) {
#pragma unroll
    for (int i = 0; i < NF; i++) {
      w2[i] = ldq(m + (int64_t)min(n, C - 1) * F, min(lane + 64 * i, nf - 1));
    }
  };
  auto get = [&](const float *s, float4 (&x)[NV]) {
#pragma unroll
    for (int i = 0; i < NV; i++) x[i] = ldq(s, min(lane + 64 * i, nv - 1));
  };
  auto dot_row = [&](const float4 (&w)[NV], const float4 (&x)[NV]) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++) s = lane + 64 * i < nv ? dot4(w[i], x[i], s) : s;
    return wave_sum(s);
  };
  // this thread's place in a slice of keys: features 4 f .. of every KEYS-th key
  const int f = threadIdx.x & (a.lanes - 1), keys = 256 / a.lanes, key = threadIdx.x / a.lanes;
  const bool has_f = 4 * f < a.head_size;
  const int64_t pitch = 3 * (int64_t)C;
  // of keys j0 + key + u KEYS of the unit's slice; the newest comes through `fresh`.  The first token of all has no earlier row: its
  // loads go to the weights (3 rows of C and more), for values that are not used.
  auto load_keys = [&](int l, int unit, int j0) {
    const int h = unit % a.heads, begin = unit / a.heads * a.slice, count = min(a.slice, a.n - begin);
    const float *p = (a.n > 1 ? a.kv + l * a.layer_stride : at(a.layer[l].wqkv)) + C + h * a.head_size + 4 * (has_f ? f : 0);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float *row = p + (int64_t)max(0, min(begin + min(j0 + u * keys + key, count - 1), a.n - 2)) * pitch;
      kk[u] = ldq(row, 0);
      vv[u] = ldq(row + C, 0);
    }
  };
#pragma unroll
  for (int r = 0; r < RA; r++) row_of(wa[r], at(a.layer[0].wqkv), gw + r * W, 3 * C);
  load_keys(0, min((int)blockIdx.x, units - 1), 0);
  row_of(wo, at(a.layer[0].wo), gw, C);
#pragma unroll 1
  for (int l = 0; l < a.layers; l++) {
    const AhDecodeLayer &w = a.layer[l];
    const uint32_t tag = a.tag + l;
    // ---- LayerNorm, q, k, v
    if (in_qkv) {
      if (meet()) return;
      float4 x[NV];
      get(xn, x);
      float *row = a.kv + l * a.layer_stride + (a.n - 1) * pitch;
      auto leave = [&](int n, float s) {
        if (lane == 0) { put(WORD_QKV + n, tag, s); row[n] = s; }
      };
#pragma unroll
      for (int r = 0; r < RA; r++) {
        const int n = gw + r * W;
        if (n < 3 * C) leave(n, dot_row(wa[r], x));
      }
      for (int n = gw + RA * W; n < 3 * C; n += W) {
        row_of(wa[0], at(w.wqkv), n, 3 * C);
        leave(n, dot_row(wa[0], x));
      }
    }
#pragma unroll
    for (int r = 0; r < RA; r++) row_of(wa[r], at(DUAL && r >= PAIRS ? w.up : w.fc1), gw + (DUAL ? r % (PAIRS ? PAIRS : 1) : r) * W, F);
    // ---- the newest query against the keys of a slice, for one head
    for (int unit = blockIdx.x; unit < units; unit += G) {
      const int h = unit % a.heads, slice = unit / a.heads, begin = slice * a.slice, count = min(a.slice, a.n - begin);
      if (meet()) return;
      const float4 none = make_float4(0.f, 0.f, 0.f, 0.f), q = has_f ? ldq(fresh[0], f) : none;
      float m = -INFINITY, sum = 0.f;
      float4 o = none;
      for (int j0 = 0; j0 < count; j0 += U * keys) {
        if (j0 > 0 || unit != (int)blockIdx.x) load_keys(l, unit, j0);
        // the group's U scores, one of them to a lane for what tanh and exp take
        float mine = 0.f;
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int j = j0 + u * keys + key;
          if (begin + j == a.n - 1) { kk[u] = ldq(fresh[1], has_f ? f : 0); vv[u] = ldq(fresh[2], has_f ? f : 0); }
          const float s = group_sum(has_f ? dot4(q, kk[u], 0.f) : 0.f, a.lanes);
          mine = (f & (U - 1)) == u ? s : mine;
        }
        mine *= a.scale;
        if (a.cap > 0.f) mine = a.cap * tanhf(mine / a.cap);
        if (j0 + (f & (U - 1)) * keys + key >= count) mine = -INFINITY;
        const float most = fmaxf(m, wave_max(mine)), old = slice_weight(m, most), p = (f & ~(U - 1)) == 0 ? slice_weight(mine, most) : 0.f;
        sum = __builtin_fmaf(sum, old, wave_sum(p));
        o.x *= old; o.y *= old; o.z *= old; o.w *= old;
        m = most;
#pragma unroll
        for (int u = 0; u < U; u++) {
          const float pu = __shfl(p, (lane & ~(a.lanes - 1)) + u, 64);
          // whatever was loaded for a key past the slice stays out: its weight is zero, and zero times an infinity is not.  (Zeros in its place
          // before the scores are made wait for the values there: 4 x 128 behind 4000 rows 137 us a token, here 133.)
          const bool in = j0 + u * keys + key < count;
          o.x = in ? __builtin_fmaf(pu, vv[u].x, o.x) : o.x; o.y = in ? __builtin_fmaf(pu, vv[u].y, o.y) : o.y;
          o.z = in ? __builtin_fmaf(pu, vv[u].z, o.z) : o.z; o.w = in ? __builtin_fmaf(pu, vv[u].w, o.w) : o.w;
        }
      }
      auto far = [&](auto step) { o.x = step(o.x); o.y = step(o.y); o.z = step(o.z); o.w = step(o.w); };
      if (a.lanes < 16) far([](float v) { return add_lane<8>(v); });
      if (a.lanes < 32) far([](float v) { return add_lane<16>(v); });
      if (a.lanes < 64) far([](float v) { return add_lane<32>(v); });
      if (lane < a.lanes && has_f) reinterpret_cast<float4 *>(part_o[wave])[lane] = o;
      if (lane == 0) { part_m[wave] = m; part_l[wave] = sum; }
      __syncthreads();
      const float most = fmaxf(fmaxf(part_m[0], part_m[1]), fmaxf(part_m[2], part_m[3]));
      float c[4];
      sum = 0.f;
#pragma unroll
      for (int v = 0; v < 4; v++) { c[v] = slice_weight(part_m[v], most); sum = __builtin_fmaf(c[v], part_l[v], sum); }
      if ((int)threadIdx.x < a.head_size) {
        float v = 0.f;
#pragma unroll
        for (int u = 0; u < 4; u++) v = __builtin_fmaf(c[u], part_o[u][threadIdx.x], v);
        put(WORD_SUMS + slice * C + h * a.head_size + threadIdx.x, tag, v);
      }
      if (threadIdx.x == 0) {
        put(WORD_TOPS + (slice * a.heads + h) * 2, tag, most);
        put(WORD_TOPS + (slice * a.heads + h) * 2 + 1, tag, sum);
      }
    }
    // ---- the slices joined, wo, the residual stream
    if (in_c) {
      if (meet()) return;
      if (meet()) return;
      float4 x[NV];
      get(joined, x);
      for (int n = gw; n < C; n += W) {
        if (n != gw) row_of(wo, at(w.wo), n, C);
        const float s = dot_row(wo, x);
        if (lane == 0) put(WORD_MID + n, tag, stream[n] + s);
      }
    }
    long_row(at(w.fc2), gw);
    // ---- LayerNorm, fc1 and its activation
    if (in_f || in_c) {
      if (meet()) return;
    }
    if (in_f) {
      float4 x[NV];
      get(xn, x);
      if constexpr (DUAL) {
        auto leave = [&](int n, float s, float t) {
          if (lane == 0) put(WORD_HID + n, tag, silu(s) * t);
        };
#pragma unroll
        for (int r = 0; r < PAIRS; r++) {
          const int n = gw + r * W;
          if (n < F) leave(n, dot_row(wa[r], x), dot_row(wa[PAIRS + r], x));
        }
        for (int n = gw + PAIRS * W; n < F; n += W) {
          row_of(wa[0], at(w.fc1), n, F);
          row_of(wa[1], at(w.up), n, F);
          leave(n, dot_row(wa[0], x), dot_row(wa[1], x));
        }
      } else {
        // a lane for each of the wave's rows: the activation is computed once
        float mine = 0.f;
#pragma unroll
        for (int r = 0; r < RA; r++)
          if (gw + r * W < F) {
            const float s = dot_row(wa[r], x);
            mine = lane == r ? s : mine;
          }
        DecodeRows c;
        c.mask = a.mask;
#pragma unroll
        for (int k = 0; k < 5; k++) c.coef[k] = at(w.coef[k]);
        const int n = gw + lane * W;
        if (lane < RA && n < F) put(WORD_HID + n, tag, activate(c, n, mine));
        for (int n = gw + RA * W; n < F; n += W) {
          row_of(wa[0], at(w.fc1), n, F);
          const float s = dot_row(wa[0], x);
          if (lane == 0) put(WORD_HID + n, tag, activate(c, n, s));
        }
      }
    }
    // of the next layer, or the first rows of the head
    const bool last = l + 1 == a.layers;
    const float *next = last ? a.head : at(a.layer[l + 1].wqkv);
    const int N = last ? a.vocab : 3 * C;
#pragma unroll
    for (int r = 0; r < RA; r++) row_of(wa[r], next, gw + r * W, N);
    // ---- fc2, the residual stream
    if (in_c) {
      if (meet()) return;
      for (int n = gw; n < C; n += W) {
        if (n != gw) long_row(at(w.fc2), n);
        float s[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NF; i++) {
          const int j = lane + 64 * i;
          s[i & 1] = j < nf ? dot4(w2[i], ldq(hid, min(j, nf - 1)), s[i & 1]) : s[i & 1];
        }
        const float t = wave_sum(s[0] + s[1]);
        if (lane == 0) put(WORD_STREAM + n, tag, mid[n] + t);
      }
    }
    const int after = last ? l : l + 1;
    if ((int)blockIdx.x < units) load_keys(after, blockIdx.x, 0);
    row_of(wo, at(a.layer[after].wo), gw, C);
  }
  // ---- the head
  if (meet()) return;
  float4 x[NV];
  get(xn, x);
  for (int n = gw; n < a.vocab; n += RA * W) {
    float4 next[RA][NV];
#pragma unroll
    for (int r = 0; r < RA; r++) row_of(next[r], a.head, n + (RA + r) * W, a.vocab);
#pragma unroll
    for (int r = 0; r < RA; r++) {
      const float s = dot_row(wa[r], x);
      if (lane == 0 && n + r * W < a.vocab) a.logits[n + r * W] = s;
#pragma unroll
      for (int i = 0; i < NV; i++) wa[r][i] = next[r][i];
    }
  }
}
__global__ __launch_bounds__(256) void k_chain_clear() {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < WORDS; i += gridDim.x * 256) chain_words[i] = 0;
}

// More results to a wave where that leaves the chip its 1000 waves or so: the row is read and normalised once for them.
template <int PRO, int NV>
void launch_rows_nv(const DecodeRows &a) {
  constexpr int MANY = NV <= 4 ? 4 : 1;
  auto go = [&](auto kfn, int r) { ah::launch_kernel(kfn, dim3((unsigned)cdiv(a.N, 4 * r)), dim3(256), 0, a); };
  if constexpr (PRO == NORM) {
    if (a.w_up) { go(k_decode_rows<NORM, NV, 1, true>, 1); return; }
    if (MANY > 1 && a.N >= 2048) { go(k_decode_rows<NORM, NV, MANY, false>, MANY); return; }
  }
  go(k_decode_rows<PRO, NV, 1, false>, 1);
}
template <int PRO>
void launch_rows(const DecodeRows &a) {
  const int nv = (int)cdiv(a.K, 256);
  if (nv <= 1) launch_rows_nv<PRO, 1>(a);
  else if (nv == 2) launch_rows_nv<PRO, 2>(a);
  else if (nv == 3) launch_rows_nv<PRO, 3>(a);
  else if (nv == 4) launch_rows_nv<PRO, 4>(a);
  else if (nv <= 8) launch_rows_nv<PRO, 8>(a);
  else launch_rows_nv<PRO, 16>(a);
}
void launch_attention(const DecodeAttention &a, int slices, int heads) {
  auto go = [&](auto kfn) { ah::launch_kernel(kfn, dim3((unsigned)slices, (unsigned)heads), dim3(256), 0, a); };
  const int quads = a.head_size / 4;
  if (quads <= 8) go(k_decode_attention<8>);
  else if (quads <= 16) go(k_decode_attention<16>);
  else go(k_decode_attention<32>);
}
int32_t check_model(const AhDecode *d) {
  AH_ARG(d != nullptr, "ah_decode: null description");
  AH_ARG(d->width > 0 && d->heads > 0 && d->width % d->heads == 0 && d->width <= MAX_WIDTH, "ah_decode: width %d in %d heads (at most %d wide)",
         d->width, d->heads, MAX_WIDTH);
  const int hs = d->width / d->heads;
  AH_ARG(hs % 8 == 0 && hs <= 128, "ah_decode: head size %d is not a multiple of 8 up to 128", hs);
  AH_ARG(d->vocab > 0 && d->layers >= 0 && d->rows > 0, "ah_decode: vocab %d, layers %d, rows %d", d->vocab, d->layers, d->rows);
  AH_ARG(d->layers == 0 || (d->ffn > 0 && d->ffn % 4 == 0), "ah_decode: ffn width %d is not a multiple of 4", d->ffn);
  AH_ARG(d->lnf_w && d->lnf_b && d->head && d->logits, "ah_decode: null operand");
  AH_ARG(aligned16(d->lnf_w | d->lnf_b | d->head), "ah_decode: operands must be 16-byte aligned");
  return AH_OK;
}
DecodeRows rows_of(const AhDecode *d, ah_ptr gain, ah_ptr bias, ah_ptr w, int n) {
  DecodeRows a = {};
  a.gain = dp<const float>(gain); a.bias = dp<const float>(bias); a.w = dp<const float>(w);
  a.N = n; a.K = d->width; a.eps = d->eps;
  return a;
}

// Where the token runs in one launch: up to 512 wide (ffn 2048), and with the layers that fit the kernel's arguments.  Wider, every phase's words
// are asked for by every workgroup at 3 to 24 KB a time, their trips through memory take 5 to 7 us instead of 2 to 3, and the rows ahead no longer
// fit the registers: 768 wide in 12 layers 430 us a token against 400 in launches.  Past 256 wide (ffn 1024) that grows with the slices of the keys,
// whose sums every workgroup joins, and up to four are taken (us a token as sampled, five launches a layer / one launch; the launches' host work
// differs that much between processes: 8 x 512 behind 17 rows 163 to 213 / 186, behind 200 165 to 207 / 195, behind 500 181 to 213 / 221, behind 900 197 to
// 224 / 237; at 256 wide 6 layers behind 900 123 to 175 / 132).  A single layer gains less than the phases of a long head lose, whose rows have few waves
// here: 1 x 256 with a vocabulary of 8000 129 / 135, 2 x 256 153 to 185 / 150.  Not inside a captured graph or a step plan, whose replays would
// bring the same tags again, nor on the side stream, where the launches of a layer are refused too.
int chain_lanes(int head_size) {
  int lanes = 8;
  while (4 * lanes < head_size) lanes *= 2;
  return lanes;
}
// keys to a slice: what the lanes hold at a time, at most 128
int chain_slice(int head_size) { return std::min(256 / chain_lanes(head_size) * CHAIN_UNITS, 128); }
int chain_quads(const AhDecode *d, int n) {
  if (d->layers > CHAIN_LAYERS || ah::step_active() || ah::capturing() || ah::on_side()) return 0;
  const int64_t nv = std::max(cdiv(d->width, 256), cdiv(d->ffn, 1024));
  if (nv > CHAIN_NV || (nv > 1 && n > 4 * chain_slice(d->width / d->heads)) || (d->layers == 1 && d->vocab > 2048)) return 0;
  return (int)nv;
}
thread_local int64_t next_ticks = SPIN_TICKS;
std::atomic<int64_t> chain_tokens{0};
int32_t launch_chain(const AhDecode *d, const AhDecodeLayer *layers, int32_t token, int32_t pos, int nv, int64_t ticks) {
  static std::atomic<uint32_t> tags{1};
  const int C = d->width, H = d->heads, hs = C / H, n = pos + 1;
  const uint32_t used = 2 * (uint32_t)d->layers;
  uint32_t tag = tags.fetch_add(used);
  if (tag > 0xf0000000u) {                      // once in 4e9 layers: no word may bear a tag that comes again
    ah::launch_kernel(k_chain_clear, dim3(64), dim3(256), 0);
    tags.store(1 + used);
    tag = 1;
  }
  DecodeChain a = {};
  for (int i = 0; i < d->layers; i++) a.layer[i] = layers[i];
  a.lnf_w = d->lnf_w; a.lnf_b = d->lnf_b;
  a.tok = dp<const float>(d->wte) + (int64_t)token * C; a.pos = dp<const float>(d->wpe) + (int64_t)pos * C;
  a.head = dp<const float>(d->head); a.kv = dp<float>(d->kv); a.logits = dp<float>(d->logits);
  a.vocab = d->vocab; a.width = C; a.heads = H; a.head_size = hs; a.ffn = d->ffn; a.layers = d->layers;
  const bool gated = (d->act & AH_DECODE_GATED) != 0;
  a.mask = gated ? 0 : d->act;
  a.n = n; a.layer_stride = (int64_t)d->rows * 3 * C;
  // slices are longer where there would be too many
  a.lanes = chain_lanes(hs);
  const int held = chain_slice(hs);
  a.slices = (int)(cdiv(n, held) < MAX_SLICES ? cdiv(n, held) : MAX_SLICES);
  a.slice = (int)cdiv(n, a.slices);
  a.slices = (int)cdiv(n, a.slice);
  a.scale = d->scale; a.cap = d->cap; a.eps = d->eps;
  const int rows = std::max(std::max(3 * C, d->ffn), std::max(d->vocab, 4 * a.slices * H));
  const unsigned grid = (unsigned)std::min<int64_t>(cdiv(rows, 4), ah::num_cus());
  auto go = [&](auto kfn) {
    a.tag = tag; a.rescue = 0; a.ticks = ticks;
    ah::launch_kernel(kfn, dim3(grid), dim3(512), 0, a);
    a.rescue = tag; a.tag = tag + (uint32_t)d->layers; a.tries = ticks < -1 ? 1 : RESCUE_TRIES;
    ah::launch_kernel(kfn, dim3(1), dim3(512), 0, a);
  };
  if (gated) { if (nv == 1) go(k_decode_chain<1, true>); else go(k_decode_chain<2, true>); }
  else { if (nv == 1) go(k_decode_chain<1, false>); else go(k_decode_chain<2, false>); }
  AH_LAUNCH_CHECK();
  chain_tokens++;
  return AH_OK;
}

}  // namespace

extern "C" {

int32_t ah_decode_next_ticks(int32_t ticks) {
  next_ticks = ticks;
  return AH_OK;
}

int32_t ah_decode_stats(int64_t *one_launch, int64_t *again) {
  AH_REQUIRE_READY();
  AH_ARG(one_launch && again, "ah_decode_stats: null result");
  if (ah::step_active() || ah::capturing()) return fail(AH_ERR_STATE, "ah_decode_stats: not inside a capture or a step plan");
  AH_HIP(hipStreamSynchronize(ah::stream()));
  uint64_t n = 0;
  AH_HIP(hipMemcpyFromSymbol(&n, HIP_SYMBOL(chain_again), sizeof(n)));
  *one_launch = chain_tokens.load();
  *again = (int64_t)n;
  return AH_OK;
}

int32_t ah_decode_head(const AhDecode *d, ah_ptr row) {
  AH_REQUIRE_READY();
  { const int32_t rc = check_model(d); if (rc != AH_OK) return rc; }
  AH_ARG(row && aligned16(row), "ah_decode_head: the row must be 16-byte aligned");
  DecodeRows a = rows_of(d, d->lnf_w, d->lnf_b, d->head, d->vocab);
  a.x = dp<const float>(row);
  a.out = dp<float>(d->logits);
  launch_rows<NORM>(a);
  AH_LAUNCH_CHECK();
  return AH_OK;
}

int32_t ah_decode(const AhDecode *d, const AhDecodeLayer *layers, int32_t token, int32_t pos) {
  const int64_t ticks = std::exchange(next_ticks, SPIN_TICKS);      // (for this token, whichever way it goes)
  AH_REQUIRE_READY();
  { const int32_t rc = check_model(d); if (rc != AH_OK) return rc; }
  AH_ARG(d->layers > 0 && layers && d->wte && d->wpe && d->kv, "ah_decode: null operand");
  AH_ARG(aligned16(d->wte | d->wpe | d->kv), "ah_decode: operands must be 16-byte aligned");
  AH_ARG(token >= 0 && token < d->vocab, "ah_decode: token %d of a vocabulary of %d", token, d->vocab);
  AH_ARG(pos >= 0 && pos < d->rows, "ah_decode: position %d of %d rows", pos, d->rows);
  AH_ARG((d->act & ~(31 | AH_DECODE_GATED)) == 0, "ah_decode: unknown activation %d", d->act);
  const bool gated = (d->act & AH_DECODE_GATED) != 0;
  for (int i = 0; i < d->layers; i++) {
    const AhDecodeLayer &l = layers[i];
    AH_ARG(l.ln1_w && l.ln1_b && l.wqkv && l.wo && l.ln2_w && l.ln2_b && l.fc1 && l.fc2 && (!gated || l.up), "ah_decode: null weight in layer %d", i);
    AH_ARG(aligned16(l.ln1_w | l.ln1_b | l.wqkv | l.wo | l.ln2_w | l.ln2_b | l.fc1 | l.fc2 | l.up), "ah_decode: weights of layer %d must be 16-byte aligned", i);
  }
  if (const int nv = chain_quads(d, pos + 1)) return launch_chain(d, layers, token, pos, nv, ticks);
  const int C = d->width, H = d->heads, n = pos + 1;
  const int slices = (int)(cdiv(n, MIN_SLICE) < MAX_SLICES ? cdiv(n, MIN_SLICE) : MAX_SLICES);
  // the residual stream, the MLP's hidden row, the slices' sums and their maxima; stream-ordered, so it may go back at once
  const int64_t hidden = (d->ffn + 3) & ~3, total = C + hidden + (int64_t)slices * (C + 2 * H);
  ah_ptr work = 0;
  { const int32_t rc = ah_alloc((uint64_t)total * 4, &work); if (rc != AH_OK) return rc; }
  float *stream = dp<float>(work), *hid = stream + C, *sums = hid + hidden;
  float2 *top = reinterpret_cast<float2 *>(sums + (int64_t)slices * C);
  for (int i = 0; i < d->layers; i++) {
    const AhDecodeLayer &l = layers[i];
    float *qkv = dp<float>(d->kv) + (int64_t)i * d->rows * 3 * C;
    DecodeRows a = rows_of(d, l.ln1_w, l.ln1_b, l.wqkv, 3 * C);
    a.x = stream; a.stream = stream;
    a.out = qkv + (int64_t)pos * 3 * C;
    if (i == 0) { a.tok = dp<const float>(d->wte) + (int64_t)token * C; a.pos = dp<const float>(d->wpe) + (int64_t)pos * C; }
    launch_rows<NORM>(a);
    DecodeAttention t = {qkv, sums, top, n, (int)cdiv(n, slices), C, C / H, d->scale, d->cap};
    launch_attention(t, slices, H);
    a = rows_of(d, 0, 0, l.wo, C);
    a.x = sums; a.top = top; a.slices = slices; a.heads = H; a.stream = stream;
    launch_rows<JOIN>(a);
    a = rows_of(d, l.ln2_w, l.ln2_b, l.fc1, d->ffn);
    a.x = stream; a.out = hid;
    if (gated) a.w_up = dp<const float>(l.up);
    else {
      a.mask = d->act;
      for (int k = 0; k < 5; k++) a.coef[k] = dp<const float>(l.coef[k]);
    }
    launch_rows<NORM>(a);
    ah::launch_kernel(k_decode_long, dim3((unsigned)C), dim3(256), 0, dp<const float>(l.fc2), hid, stream, d->ffn);
  }
  int32_t rc = AH_OK;
  {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = ah::hip_fail(e, __func__);
    else ah::count_op();
  }
  if (rc == AH_OK) rc = ah_decode_head(d, work);
  const int32_t rf = ah_free(work);
  return rc ? rc : rf;
}

}  // extern "C"
