// The FP64 quotients and roots without range handling (fx_device.hpp), one
// operand pair a thread, for tests/test_gpu_fast_division.py: out holds
// recip_rn(y), quot(x, y), quot_r(x, y, recip_rn(y)) and sqrt_fast(|y|), n each.
#include <hip/hip_runtime.h>

#include "fx_device.hpp"

namespace {
__global__ void k_div(const double* __restrict__ x, const double* __restrict__ y, long n,
                      double* __restrict__ out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double r = fx::recip_rn(y[i]);
  out[i] = r;
  out[n + i] = fx::quot(x[i], y[i]);
  out[2 * n + i] = fx::quot_r(x[i], y[i], r);
  out[3 * n + i] = fx::sqrt_fast(fabs(y[i]));
}
}  // namespace

// x, y: n doubles on the device; out: 4 n.  Waits; returns 0, or HIP's error.
extern "C" int fx_test_div(const double* x, const double* y, long n, double* out) {
  if (n <= 0 || n > (1L << 30)) return 1;
  hipLaunchKernelGGL(k_div, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, nullptr, x, y, n, out);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess ? (int)e : (int)hipDeviceSynchronize();
}
