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

// Rows per band: 4 halo rows each, but a wave walks its band row after row.  The
// longest of 32, 16, 8 that leaves 3 waves per SIMD (3072).  us per step, walking
// sweeps with 8 / 16 / 32 rows: 1531x1021 210 / 218 / 230, 2048^2 mixed 421 / 418 / 439,
// 3072x1024 three materials mixed 639 / 630 / 668, 4096^2 1760 / 1761 / 1750.
int sweepWalkRows(long nx, long ny) {
  for (int rows : {32, 16})
    if ((nx + 63) / 64 * ((ny + rows - 1) / rows) >= 3072) return rows;
  return 8;
}

// launch grid of the walking y sweeps (256-thread blocks of 4 waves)
dim3 sweepWalkGrid(long nx, long ny, int rows) {
  const long waves = (nx + 63) / 64 * ((ny + rows - 1) / rows);
  return dim3((unsigned)((waves + 3) / 4));
}

}  // namespace mhy
