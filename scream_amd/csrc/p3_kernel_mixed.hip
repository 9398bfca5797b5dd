// Mixed-precision variants (FP32 bulk process rates, FP64 saturation, limiters,
// updates and sedimentation fluxes; with P3_SED_LPC: the sedimentation launches
// on that many lanes per column).
#include "p3_launch.hpp"
namespace p3d {
#define REAL float
#define SED_CAT(lpc) sed_launch_mixed_##lpc
#define SED_NAME(lpc) SED_CAT(lpc)
#ifdef P3_SED_LPC
#include "p3_sed_variants.inc"
#else
SedLaunch SED_NAME(16)(), SED_NAME(32)(), SED_NAME(64)();
#define LAUNCH_NAME launch_p3_mixed
#define LAUNCH_BATCH_NAME launch_p3_batch_mixed
#define OCC_NAME occupancy_p3_mixed
#include "p3_kernel_variants.inc"
// One thread; the expressions of part2_level.
__global__ void p3_rain_gamma_kernel(float mu_r, float* d) {
  d[0] = m_tgamma(mu_r + 1.f);
  d[1] = m_tgamma(mu_r + 2.f);
  d[2] = m_log(m_tgamma(7.f + mu_r));
  d[3] = m_log(m_tgamma(4.f + mu_r));
}
hipError_t rain_gamma_mixed(float mu, float* d, RainGamma* out) {
  float v[4];
  hipLaunchKernelGGL(p3_rain_gamma_kernel, dim3(1), dim3(1), 0, nullptr, mu, d);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpy(v, d, sizeof(v), hipMemcpyDeviceToHost);
  if (e == hipSuccess) *out = {mu, v[0], v[1], v[2], v[3]};
  return e;
}
#endif
}  // namespace p3d
