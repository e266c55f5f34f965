// Error state and version of the C ABI (include/trnsparse_hip.h).
#include <stdarg.h>
#include <stdio.h>

#include "common.h"

namespace tsp {

static thread_local char g_err[1024] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int check_hip(hipError_t e, const char* what) {
  if (e == hipSuccess) return TSP_OK;
  return fail(TSP_EHIP, "%s: %s (%s)", what, hipGetErrorString(e), hipGetErrorName(e));
}

int check_launch(const char* what) { return check_hip(hipGetLastError(), what); }

// rows of n units, `ld` units apart. Bound by the launch for small fills and by
// the writes for large ones.
template <typename U>
__global__ __launch_bounds__(256) void zero_fill_kernel(U* __restrict__ p, int64_t rows, int64_t ld, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = blockIdx.y; r < rows; r += gridDim.y)
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[r * ld + i] = U{};
}

int zero_fill_rows(void* p, int64_t rows, int64_t ld, int64_t bytes, hipStream_t st) {
  if (rows <= 0 || bytes <= 0) return TSP_OK;
  auto go = [&](auto unit) {
    typedef decltype(unit) U;
    const int64_t n = bytes / (int64_t)sizeof(U), gy = rows < 1024 ? rows : 1024, most = 4096 / gy;
    const int64_t gx = ceil_div(n, 256) < most ? ceil_div(n, 256) : most;
    hipLaunchKernelGGL(zero_fill_kernel<U>, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, st, (U*)p, rows,
                       ld / (int64_t)sizeof(U), n);
    return check_launch("zero_fill launch");
  };
  // the widest store that the address, the row stride and the row length allow
  const uint64_t all = (uint64_t)(uintptr_t)p | (uint64_t)bytes | (rows > 1 ? (uint64_t)ld : 0);
  if (all % 16 == 0) return go(u32x4{});
  if (all % 4 == 0) return go(uint32_t{});
  return go(uint8_t{});
}

int zero_fill(void* p, int64_t bytes, hipStream_t st) { return zero_fill_rows(p, 1, 0, bytes, st); }

}  // namespace tsp

extern "C" int tsp_version(void) { return 100; }

extern "C" const char* tsp_last_error(void) { return tsp::g_err; }
