// p3_launch.hpp -- host-side entry points of the compiled kernel variants.
#pragma once

#include <hip/hip_runtime.h>

#include "p3_batch.hpp"

namespace p3d {

// Shape of one step's launches: the lanes per column of the sedimentation
// kernels (16, 32 or 64), of the liquid group (cloud, rain) and of the ice
// group; each lane holds L = ceil(nlev / lanes) levels (at most 8), 4 wavefronts
// per block (the batched form runs both groups of a set on lpc).  Parts 1 to 3 run one
// thread per (level, column) on the pointwise tiles.
struct Shape {
  int lpc, lpc_ice;
};

// Largest levels-per-lane count of the sedimentation kernel.
constexpr int kMaxLevelsPerLane = 8;
// Wavefronts per block of the sedimentation kernel.
#ifndef P3_SED_WAVES
#define P3_SED_WAVES 4
#endif
constexpr int kSedWaves = P3_SED_WAVES;

// Levels per lane the sedimentation kernel is instantiated with for nlev
// levels on lpc lanes (0 if nlev does not fit).
inline int sed_levels_per_lane(int nlev, int lpc) {
  const int l = (nlev + lpc - 1) / lpc;
  if (l <= 6) return l < 1 ? 1 : l;
  return l <= kMaxLevelsPerLane ? kMaxLevelsPerLane : 0;
}

// A second stream for the liquid group's sedimentation kernel: with one, that
// kernel runs beside the ice group's (they touch disjoint fields), forked from
// s after part 2 (event fork) and joined back into s before part 3 (event join).
struct SedFork {
  hipStream_t side;
  hipEvent_t fork, join;
};

// hipErrorInvalidValue for a shape that is not compiled in.
// `between` (optional) is recorded on s after part 2, before sedimentation;
// `fork` (optional) runs the two sedimentation kernels concurrently.
hipError_t launch_p3_fp64(const KParams& p, const Shape& sh, hipStream_t s, hipEvent_t between = nullptr,
                          const SedFork* fork = nullptr);
hipError_t launch_p3_mixed(const KParams& p, const Shape& sh, hipStream_t s, hipEvent_t between = nullptr,
                           const SedFork* fork = nullptr);

// RainGamma of the mixed form for the shape parameter mu, in its own arithmetic on
// the current device; d: four floats of device memory for the result.
hipError_t rain_gamma_mixed(float mu, float* d, RainGamma* out);

// ---- batched form (p3_batch.hpp)
// Sets whose sedimentation runs on the same lanes per column and levels per lane.
struct SedClass {
  int lpc, L;
  const KParams* sets;  // device array
  const int* first;     // device array, nsets + 1 entries
  int nsets;
  int total;            // virtual blocks per species group (first[nsets])
  int grid;             // blocks (one per virtual block, or a persistent grid)
};
constexpr int kMaxSedClasses = 3 * kMaxLevelsPerLane;
// Streams beside the batch's own for its second and later classes.
constexpr int kSideStreams = 3;
// The sedimentation launches on one lanes-per-column count.
struct SedLaunch {
  hipError_t (*single)(const KParams& p, int group, int L, hipStream_t s);  // one species group
  hipError_t (*fused)(const KParams& p, int L, hipStream_t s);              // both groups, one launch
  hipError_t (*batch)(const SedClass& c, hipStream_t s);
  hipError_t (*occupancy)(int L, int* blocks);  // resident blocks per CU of the batched kernels
};
struct BatchPlan {
  const KParams* sets;  // device array, all sets (pointwise launches)
  const int* first;     // device array, nsets + 1 entries: pointwise tiles (parts 1 to 3)
  int nsets;
  int ordered;          // some set's sedimentation takes the columns in p3_order_batch's order
  int order_blocks;     // blocks of p3_order_batch per set
  int track;            // some set keeps its column status words (KParams::track)
  int grid;             // blocks of the pointwise launches
  int total;            // pointwise virtual blocks (first[nsets]); grid >= total: one block each, no loop
  int nclass;
  SedClass cls[kMaxSedClasses];
  // with side streams (NULL: none), the classes run side by side, forked from
  // the batch's stream after parts 1 and 2 and joined before part 3
  hipStream_t side[kSideStreams];
  hipEvent_t fork, join[kSideStreams];
};
hipError_t launch_p3_batch_fp64(const BatchPlan& b, hipStream_t s);
hipError_t launch_p3_batch_mixed(const BatchPlan& b, hipStream_t s);
// Resident blocks per CU of the batched kernels for this shape (occupancy API).
hipError_t occupancy_p3_fp64(int lpc, int L, int* blocks, int* blocks_sed);
hipError_t occupancy_p3_mixed(int lpc, int L, int* blocks, int* blocks_sed);

}  // namespace p3d
