// The host side of the fp32 products without a GPU: links with the built gemm_f32 object in place of the runtime, and prints for every
// line "M N K layout epilogue refuse lda" on the standard input (refuse: 1 device memory is refused, 2 the second launch fails, 3 the
// caller wants one piece) what gemm_f32 would launch:
//   return code | last kernel noted | slices noted | blocks outstanding | launch ...    with launch = grid x * threads, K of a slice
// or "join" for the launch that adds up the slices
// Built for the host only (hipcc --cuda-host-only); no HIP runtime is linked.
#include "../alpha2_amd/csrc/gemm_common.h"
#include <cstdarg>
#include <cstdio>
#include <string>

static std::string g_kernel, g_launches;
static int g_split = 0, g_live = 0, g_refuse = 0, g_count = 0;

namespace ah {
void launch_raw(const void *, dim3 grid, dim3 block, unsigned, void **args, const uint32_t *sizes, int) {
  g_count++;
  if (sizes[0] != sizeof(GemmArgs)) { g_launches += " join"; return; }
  const GemmArgs &g = *(const GemmArgs *)args[0];
  char s[96];
  snprintf(s, sizeof s, " %llu,%d", (unsigned long long)grid.x * block.x, g.nsplit > 1 ? g.ksplit : g.K);
  g_launches += s;
}
int32_t splitk_reduce(const float *, float *, int, int, int, int64_t, bool) { g_launches += " join"; return AH_OK; }
void note_gemm_kernel(const char *fmt, ...) {
  char s[96];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(s, sizeof s, fmt, ap);
  va_end(ap);
  g_kernel = s;
}
void note_gemm_split(int n) { g_split = n; }
int num_cus() { return 256; }
void count_op() {}
int32_t hip_fail(hipError_t, const char *) { return AH_ERR_HIP; }
}  // namespace ah
extern "C" {
int32_t ah_alloc(uint64_t, ah_ptr *out) {
  if (g_refuse == 1) return AH_ERR_OOM;
  g_live++;
  *out = 1 << 20;
  return AH_OK;
}
int32_t ah_free(ah_ptr) { g_live--; return AH_OK; }
hipError_t hipGetLastError() { return g_refuse == 2 && g_count > 1 ? hipErrorLaunchFailure : hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { static void *handle; return &handle; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, uint3 *, uint3 *, dim3 *, dim3 *, int *) {}
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
}

int main() {
  long long m, n, k, lda;
  int layout, epi, refuse;
  while (scanf("%lld %lld %lld %d %d %d %lld", &m, &n, &k, &layout, &epi, &refuse, &lda) == 7) {
    ah::GemmArgs g{};
    g.M = (int)m; g.N = (int)n; g.K = (int)k;
    g.lda = lda ? lda : layout == AH_GEMM_TN ? m : k;
    g.ldb = layout == AH_GEMM_NT ? k : n;
    g.ldc = n;
    g.epi = epi; g.ksplit = (int)k; g.nsplit = refuse == 3 ? 0 : 1;
    g_kernel = g_launches = "";
    g_split = -1; g_live = 0; g_refuse = refuse; g_count = 0;
    const int rc = ah::gemm_f32(g, layout, 1, AH_F32, 1, 1, 1);
    printf("%d|%s|%d|%d|%s\n", rc, g_kernel.c_str(), g_split, g_live, g_launches.c_str());
  }
  return 0;
}
