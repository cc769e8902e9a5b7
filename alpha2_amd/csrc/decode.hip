// One token through the model, from the keys and values that earlier tokens left (packages/train/src/sample.ts:36-198 runs the whole
// context again for each new token; a causal row depends on the rows before it through their keys and values only).
//
// A single row makes every product a matrix times a vector: nothing is used twice, so there is no tile to share and the bound is the
// weights read once (4 bytes for 2 operations) - where a launch is long enough to feel it.  At the sizes sampled in earnest (256 to
// 1024 wide) a matrix is 0.3 to 12 MB, a microsecond or two of the chip, and what a token takes is the chain of dependent launches.
// So the launches are few, five a layer, each does the small work in front of its product itself, and each asks for its weights before
// anything it has to wait for:
//   k_decode_rows<NORM>  LayerNorm (the first one of all adds the two embeddings) + q, k, v into the row of the cache; + fc1 and its
//                        activation (gate and up together); + the head.  Every wave normalises the row again, in registers.
//   k_decode_attention   keys in slices of at least 64, one workgroup to a slice and head
//   k_decode_rows<JOIN>  joins the slices (softmax weights of the slices' maxima) in LDS + wo + the residual stream
//   k_decode_long        fc2 + the residual stream: long rows, few of them, so four waves to a row
// 64 tokens from a 6 x 256 model 56.0 -> 11.5 ms, 24 tokens behind a prompt of 480 from the GPT-2-small shape 59.9 -> 12.6 (each with
// the pass over the finished sequence that follows).  A launch takes 2.9 to 5.7 us there and the next one starts about 1 us later.
#include "common.h"
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

enum { NORM = 0, JOIN = 1 };
// A wave computes R neighbouring results (DUAL: R of the gate and R of the up matrix).  NV: float4 per lane of a row, K <= 256 NV.
template <int PRO, int NV, int R, bool DUAL>
__global__ __launch_bounds__(256) void k_decode_rows(DecodeRows a) {
  constexpr int ROWS = DUAL ? 2 * R : R;
  __shared__ __attribute__((aligned(16))) float joined[PRO == JOIN ? 256 * NV : 4];
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
    // eight slices at a time, all asked for at once (one after the other they took 10 of 13 us at 768 wide with 8 slices)
    const int head_size = a.K / a.heads;
#pragma unroll(NV <= 4 ? NV : 1)
    for (int i = 0; i < NV; i++) {
      const int k = min(threadIdx.x + 256 * i, a.K - 1), h = k / head_size;
      float most = -INFINITY, sum = 0.f, v = 0.f;
      for (int s0 = 0; s0 < a.slices; s0 += 8) {
        float2 t[8];
        float y[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int s = min(s0 + u, a.slices - 1);
          t[u] = a.top[s * a.heads + h];
          y[u] = a.x[(int64_t)s * a.K + k];
        }
        float top = most;
#pragma unroll
        for (int u = 0; u < 8; u++) top = fmaxf(top, t[u].x);
        const float old = most == -INFINITY ? 0.f : expf(most - top);
        sum *= old;
        v *= old;
        most = top;
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const float c = s0 + u >= a.slices || t[u].x == -INFINITY ? 0.f : expf(t[u].x - most);
          sum = __builtin_fmaf(c, t[u].y, sum);
          v = s0 + u < a.slices ? __builtin_fmaf(c, y[u], v) : v;
        }
      }
      joined[k] = v / sum;
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
// 256 / G keys at a time; each group of lanes keeps its own running maximum, and the groups are joined at the end.
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
  for (int j0 = key; j0 < count; j0 += KEYS * U) {
    float4 k[U], v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float *p = ks + min(j0 + u * KEYS, count - 1) * pitch;
      k[u] = ldq(p, 0);
      v[u] = ldq(p + a.width, 0);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      float s = in ? dot4(q, k[u], 0.f) : 0.f;
#pragma unroll
      for (int d = 1; d < G; d <<= 1) s += __shfl_xor(s, d, 64);
      s *= a.scale;
      if (a.cap > 0.f) s = a.cap * tanhf(s / a.cap);
      if (j0 + u * KEYS < count) {
        const float most = s > m ? s : (m >= s ? m : s);        // NaN stays
        const float old = m == -INFINITY ? 0.f : expf(m - most), p = s == -INFINITY ? 0.f : expf(s - most);
        l = __builtin_fmaf(l, old, p);
        o.x = __builtin_fmaf(o.x, old, p * v[u].x); o.y = __builtin_fmaf(o.y, old, p * v[u].y);
        o.z = __builtin_fmaf(o.z, old, p * v[u].z); o.w = __builtin_fmaf(o.w, old, p * v[u].w);
        m = most;
      }
    }
  }
  // the groups of a wave, then the waves; -inf is a group without a key
  auto weight = [](float m, float most) { return m == -INFINITY ? 0.f : expf(m - most); };
#pragma unroll
  for (int d = G; d < 64; d <<= 1) {
    const float om = __shfl_xor(m, d, 64), ol = __shfl_xor(l, d, 64);
    const float4 oo = make_float4(__shfl_xor(o.x, d, 64), __shfl_xor(o.y, d, 64), __shfl_xor(o.z, d, 64), __shfl_xor(o.w, d, 64));
    const float most = fmaxf(m, om), c = weight(m, most), e = weight(om, most);
    l = l * c + ol * e;
    o = make_float4(o.x * c + oo.x * e, o.y * c + oo.y * e, o.z * c + oo.z * e, o.w * c + oo.w * e);
    m = most;
  }
  if (lane < G) {
    reinterpret_cast<float4 *>(all_o[wave])[lane] = o;
    if (lane == 0) { all_m[wave] = m; all_l[wave] = l; }
  }
  __syncthreads();
  const float most = fmaxf(fmaxf(all_m[0], all_m[1]), fmaxf(all_m[2], all_m[3]));
  float c[4], sum = 0.f;
#pragma unroll
  for (int w = 0; w < 4; w++) { c[w] = weight(all_m[w], most); sum = __builtin_fmaf(c[w], all_l[w], sum); }
  for (int d = threadIdx.x; d < a.head_size; d += 256) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) v = __builtin_fmaf(c[w], all_o[w][d], v);
    a.sums[(int64_t)blockIdx.x * a.width + h * a.head_size + d] = v;
  }
  if (threadIdx.x == 0) a.top[blockIdx.x * gridDim.y + h] = make_float2(most, sum);
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
  if (quads <= 2) go(k_decode_attention<2>);
  else if (quads <= 4) go(k_decode_attention<4>);
  else if (quads <= 8) go(k_decode_attention<8>);
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

}  // namespace

extern "C" {

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
