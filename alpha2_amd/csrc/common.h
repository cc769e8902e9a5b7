// Shared host/device helpers for libalpha_hip (gfx950 only, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>
#include <stddef.h>
#include <tuple>
#include <utility>
#include "../../include/alpha_hip.h"

namespace ah {

// ---- host-side context (defined in runtime.hip) -------------------------------------------------
hipStream_t stream();
bool        ready();
bool        on_side();              // between ah_side_begin and ah_side_end, where nothing may be allocated
int32_t     fail(int32_t code, const char *fmt, ...);
int32_t     hip_fail(hipError_t e, const char *what);
void        count_op();
int         num_cus();
// Scratch for two-stage reductions: a library-owned device buffer of at least `bytes` bytes that stays
// valid until the next call that asks for scratch on the same stream (calls are stream-ordered).  There is ONE buffer,
// ordered by the main stream: between ah_side_begin and ah_side_end it is refused (nullptr), as is growing it while a
// graph or step plan exists.
void       *scratch(size_t bytes);
int         current_device();                     // the device ah_init was called with
int32_t     static_partials_init(int device);     // reduce.hip: device address of its static scratch array (called by ah_init)
void        gemm_plans_forget();                  // gemm.hip: every grouped-GEMM plan id becomes unknown (called by ah_shutdown)

// Every kernel of the library is launched through launch_kernel(): the arguments are converted to the kernel's parameter
// types and handed, as an array of pointers to them, to launch_raw (runtime.hip).  Outside a step plan that is
// hipLaunchKernel on the library stream.  Inside one (ah_step_begin .. ah_step_end) the launch is recorded into the
// stream capture, or -- when a plan exists -- compared with the plan's next kernel node: same kernel, same grid means
// "skip, the graph will run it", with the node's parameters rewritten if any argument differs.
void launch_raw(const void *func, dim3 grid, dim3 block, unsigned shmem, void **args, const uint32_t *sizes, int nargs);
template <class... KArgs, class... Args, size_t... I>
inline void launch_impl(void (*kernel)(KArgs...), dim3 grid, dim3 block, unsigned shmem, std::index_sequence<I...>, Args &&...args) {
  std::tuple<KArgs...> vals{static_cast<KArgs>(std::forward<Args>(args))...};
  void *ptrs[sizeof...(KArgs) + 1] = {(void *)&std::get<I>(vals)..., nullptr};
  const uint32_t sizes[sizeof...(KArgs) + 1] = {(uint32_t)sizeof(KArgs)..., 0u};
  launch_raw(reinterpret_cast<const void *>(kernel), grid, block, shmem, ptrs, sizes, (int)sizeof...(KArgs));
}
template <class... KArgs, class... Args>
inline void launch_kernel(void (*kernel)(KArgs...), dim3 grid, dim3 block, unsigned shmem, Args &&...args) {
  static_assert(sizeof...(KArgs) == sizeof...(Args), "kernel argument count");
  launch_impl(kernel, grid, block, shmem, std::index_sequence_for<KArgs...>{}, std::forward<Args>(args)...);
}
// A point where the host needs the stream's results or touches it outside a kernel launch (download, sync, events):
// inside a step plan the work recorded so far is launched first.  Returns AH_OK or an error code.
int32_t step_boundary(const char *what);
bool    step_active();
bool    capturing();                              // between ah_graph_begin and ah_graph_end

#define AH_REQUIRE_READY() do { if (!ah::ready()) return ah::fail(AH_ERR_STATE, "%s: ah_init has not been called", __func__); } while (0)
#define AH_HIP(expr) do { hipError_t _e = (expr); if (_e != hipSuccess) return ah::hip_fail(_e, #expr); } while (0)
#define AH_ARG(cond, ...) do { if (!(cond)) return ah::fail(AH_ERR_ARG, __VA_ARGS__); } while (0)
#define AH_LAUNCH_CHECK() do { hipError_t _e = hipGetLastError(); if (_e != hipSuccess) return ah::hip_fail(_e, __func__); ah::count_op(); } while (0)

template <class T> static inline T *dp(ah_ptr p) { return reinterpret_cast<T *>(static_cast<uintptr_t>(p)); }
static inline bool aligned16(ah_ptr p) { return (p & 15u) == 0; }
static inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- device helpers -----------------------------------------------------------------------------
typedef __hip_bfloat16 bf16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
// f32 -> bf16, round-to-nearest-even (v_cvt_pk_bf16_f32 on gfx950)
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2_t v;
  v[0] = (__bf16)lo; v[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) { return (uint16_t)(pack_bf16x2(f, 0.f) & 0xffffu); }

template <class T> struct Io;
template <> struct Io<float> {
  static __device__ __forceinline__ float ld(const float *p, size_t i) { return p[i]; }
  static __device__ __forceinline__ void  st(float *p, size_t i, float v) { p[i] = v; }
};
template <> struct Io<uint16_t> {   // bf16 storage
  static __device__ __forceinline__ float ld(const uint16_t *p, size_t i) { return bf16_bits_to_f32(p[i]); }
  static __device__ __forceinline__ void  st(uint16_t *p, size_t i, float v) { p[i] = f32_to_bf16_bits(v); }
};

// What lane ^ O holds; every lane of the wave takes part.  Rows of 16 and halves are exchanged by v_permlane16/32_swap, the rest is moved by DPP: a step
// of a reduction is one or two vector instructions, where __shfl_xor is a trip through LDS (ds_bpermute, 100 cycles and more), and reductions
// along a row are what a short row kernel waits for (same bits; the step of 2 layers x 128 at 2 x 64 tokens 294 -> 289 us, of
// 24 x 1024 at 4 x 8 x 1024 no more than two runs differ).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_moved(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true); }
template <int O>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32, "one bit of the lane");
  if constexpr (O == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);      // the lower halves, the upper halves
    return threadIdx.x & 32 ? r[0] : r[1];
  } else if constexpr (O == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);      // the even rows, the odd rows
    return threadIdx.x & 16 ? r[0] : r[1];
  } else if constexpr (O == 8) return dpp_moved<0x128>(v);                    // a row turned by eight
  else if constexpr (O == 4) return dpp_moved<0x1b>(dpp_moved<0x141>(v));     // eight lanes mirrored, then each four of them
  else if constexpr (O == 2) return dpp_moved<0x4e>(v);
  else return dpp_moved<0xb1>(v);
}
template <int O>
__device__ __forceinline__ float lane_xor(float v) { return __uint_as_float(lane_xor<O>(__float_as_uint(v))); }
template <int O>
__device__ __forceinline__ double lane_xor(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, (uint64_t)lane_xor<O>((uint32_t)(u >> 32)) << 32 | lane_xor<O>((uint32_t)u));
}
// v and what lane ^ O holds, in an order that both lanes share: for sums and maxima, which do not ask which is whose
template <int O>
__device__ __forceinline__ float2 lane_pair(float v) {
  if constexpr (O == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
  } else if constexpr (O == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
  } else return make_float2(v, lane_xor<O>(v));
}
template <int O> __device__ __forceinline__ float add_lane(float v) { const float2 p = lane_pair<O>(v); return p.x + p.y; }
template <int O> __device__ __forceinline__ float max_lane(float v) { const float2 p = lane_pair<O>(v); return fmaxf(p.x, p.y); }

// over G neighbours (a power of two), the near ones first
template <int G>
__device__ __forceinline__ float near_sum(float v) {
  if constexpr (G > 1) v = add_lane<1>(v);
  if constexpr (G > 2) v = add_lane<2>(v);
  if constexpr (G > 4) v = add_lane<4>(v);
  if constexpr (G > 8) v = add_lane<8>(v);
  if constexpr (G > 16) v = add_lane<16>(v);
  if constexpr (G > 32) v = add_lane<32>(v);
  return v;
}
// wave64 reductions, the far lanes first.  (In the step of 4 a row of 16 holds its eight sums twice, so turning it by four does.)
__device__ __forceinline__ float wave_sum(float v) {
  v = add_lane<8>(add_lane<16>(add_lane<32>(v)));
  v += __uint_as_float(dpp_moved<0x124>(__float_as_uint(v)));
  return add_lane<1>(add_lane<2>(v));
}
__device__ __forceinline__ double wave_sum_d(double v) {
  v += lane_xor<32>(v); v += lane_xor<16>(v); v += lane_xor<8>(v); v += lane_xor<4>(v); v += lane_xor<2>(v); v += lane_xor<1>(v);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  v = max_lane<8>(max_lane<16>(max_lane<32>(v)));
  v = fmaxf(v, __uint_as_float(dpp_moved<0x124>(__float_as_uint(v))));
  return max_lane<1>(max_lane<2>(v));
}

// tanh-approximation GELU and its derivative (cpu_ref.ts:422-427; ops.ts:405-417) on the gate
// s = sigmoid(2u) = (1 + tanh u) / 2 with u = sqrt(2/pi) (x + 0.044715 x^3):  gelu(x) = x s and
// gelu'(x) = s + x s (1 - s) 2u'.  Two hardware transcendentals, no branches, absolute error at fp32 rounding level; a
// value + derivative pair costs 9 simple operations (the epilogues of the big GEMM tiles run one wave per SIMD, where
// every instruction costs 4 cycles, and cannot afford libm's tanhf: its register footprint on top of 256 live
// accumulators spills).
__device__ __forceinline__ float gelu_gate_s(float x, float x2) {
  const float k2 = 0.7978845608028654f * 2.0f * 1.4426950408889634f;      // 2 sqrt(2/pi) log2(e)
  float z = x * __builtin_fmaf(x2, -k2 * 0.044715f, -k2);
  return __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(z) + 1.0f);
}
__device__ __forceinline__ float gelu_f(float x) { return x * gelu_gate_s(x, x * x); }
// value and derivative from one gate evaluation
__device__ __forceinline__ void gelu_both_f(float x, float &val, float &grad) {
  const float k = 0.7978845608028654f;
  float x2 = x * x, s = gelu_gate_s(x, x2);
  float h = x * s;
  float d = __builtin_fmaf(x2, 6.0f * k * 0.044715f, 2.0f * k);           // 2 du/dx
  val = h;
  grad = __builtin_fmaf(h * d, 1.0f - s, s);
}
__device__ __forceinline__ float gelu_grad_f(float x) {
  float v, d;
  gelu_both_f(x, v, d);
  return d;
}
// gelu' is 1 / 0 beyond +-40 to the last bit; evaluated there, x^3 does not overflow f32 as it would from 7e12 on (the reference
// computes in f64, ops.ts:401-419).  NaN and the infinities go through as they are (the reference's formula gives NaN for both: 0 x inf).
__device__ __forceinline__ float gelu_grad_any_f(float x) {
  const float ax = fabsf(x);
  return gelu_grad_f(ax > 40.f && ax <= 3.402823466e38f ? copysignf(40.f, x) : x);
}

}  // namespace ah
