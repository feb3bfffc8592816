// Instantiations of the column-walking y sweeps (sweep_walk.hpp): options at
// run time; the launch grid.
#include "sweep_walk.hpp"

namespace mhy {

#define MHY_SWEEP_WALK_INST(R, M, PP) \
  template __global__ void k_sweep_walk<R, M, PP, RunOpts>(KPT<R>); \
  template __global__ void k_sweep_walk_batch<R, M, PP, false>(BatchLaunchT<R>); \
  template __global__ void k_sweep_walk_batch<R, M, PP, true>(BatchLaunchT<R>);
#define MHY_SWEEP_WALK_INST_R(R) \
  MHY_SWEEP_WALK_INST(R, 1, false) \
  MHY_SWEEP_WALK_INST(R, 1, true) \
  MHY_SWEEP_WALK_INST(R, 2, false) \
  MHY_SWEEP_WALK_INST(R, 2, true) \
  MHY_SWEEP_WALK_INST(R, 3, false) \
  MHY_SWEEP_WALK_INST(R, 3, true)
MHY_SWEEP_WALK_INST_R(double)
MHY_SWEEP_WALK_INST_R(float)
#undef MHY_SWEEP_WALK_INST_R
#undef MHY_SWEEP_WALK_INST

// launch grid of the walking y sweeps (256-thread blocks of 4 waves)
dim3 sweepWalkGrid(long nx, long ny) {
  const long waves = (nx + 63) / 64 * ((ny + kWalkRows - 1) / kWalkRows);
  return dim3((unsigned)((waves + 3) / 4));
}

}  // namespace mhy
