// FP64 drop-in variants of the P3 kernels (with P3_SED_LPC: the sedimentation
// launches on that many lanes per column).
#include "p3_launch.hpp"
namespace p3d {
#define REAL double
#define SED_CAT(lpc) sed_launch_fp64_##lpc
#define SED_NAME(lpc) SED_CAT(lpc)
#ifdef P3_SED_LPC
#include "p3_sed_variants.inc"
#else
SedLaunch SED_NAME(16)(), SED_NAME(32)(), SED_NAME(64)();
#define LAUNCH_NAME launch_p3_fp64
#define LAUNCH_BATCH_NAME launch_p3_batch_fp64
#define OCC_NAME occupancy_p3_fp64
#include "p3_kernel_variants.inc"
#endif
}  // namespace p3d
