// p3_math_device.hip -- the device forms of scream_amd/csrc/p3_math.h over arrays, for
// the tests that compare them with the CPU's bits (test infrastructure, never the product).
#include <hip/hip_runtime.h>

#include "../scream_amd/csrc/p3_math.h"

namespace {
// 0 to 7 as p3o_elementary (p3_oracle.c); 8 to 11 the divisions; 12 log10_pos;
// 13 x^y from log x
__global__ void eval(int fn, int n, const double* x, const double* y, double* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double a = x[i], b = y[i];
  double r = 0;
  switch (fn) {
    case 0: r = p3m_exp(a); break;
    case 1: r = p3m_log(a); break;
    case 2: r = p3m_log10(a); break;
    case 3: r = p3m_pow(a, b); break;
    case 4: r = p3m_cbrt(a); break;
    case 5: r = p3m_tgamma(a); break;
    case 6: r = p3m_expm1(a); break;
    case 7: r = p3m_tanh(a); break;
    case 8: r = p3m_div(a, b); break;
    case 9: r = p3m_div_inf(a, b); break;
    case 10: r = p3m_div_any(a, b); break;
    case 11: r = p3m_div_n(a, b); break;
    case 12: r = p3m_log10_pos(a); break;
    case 13: {
      double h, l;
      p3m_log_core(a, &h, &l);
      r = p3m_pow_log(h, l, b);
    }
  }
  out[i] = r;
}
}  // namespace

// Host arrays of n values; 0 on success.
extern "C" int p3md_eval(int fn, int n, const double* x, const double* y, double* out) {
  if (fn < 0 || fn > 13 || n <= 0) return 1;
  double* d = nullptr;
  const size_t bytes = (size_t)n * sizeof(double);
  hipError_t e = hipMalloc((void**)&d, 3 * bytes);
  if (e == hipSuccess) e = hipMemcpy(d, x, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(d + n, y, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(eval, dim3((n + 255) / 256), dim3(256), 0, nullptr, fn, n, d, d + n, d + 2 * (size_t)n);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(out, d + 2 * (size_t)n, bytes, hipMemcpyDeviceToHost);
  (void)hipFree(d);
  return e == hipSuccess ? 0 : 2;
}

// The CPU forms of 12 and 13 (the others are p3o_elementary's and IEEE divisions).
extern "C" double p3md_host(int fn, double a, double b) {
  if (fn == 12) return p3m_log10_pos(a);
  double h, l;
  p3m_log_core(a, &h, &l);
  return p3m_pow_log(h, l, b);
}
