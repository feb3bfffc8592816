// Instantiations of the wave-strip sweeps (sweep_wave.hpp): options at run time,
// mixed form.
#include "sweep_wave.hpp"

namespace mhy {

#define MHY_SWEEP_WAVE_INST(R, M, PP) \
  template __global__ void k_sweep_wave<R, M, PP, true, RunOpts>(KPT<R>); \
  template __global__ void k_sweep_wave<R, M, PP, false, RunOpts>(KPT<R>); \
  template __global__ void k_sweep_wave_batch<R, M, PP, true, false, RunOpts>(BatchLaunchT<R>); \
  template __global__ void k_sweep_wave_batch<R, M, PP, false, false, RunOpts>(BatchLaunchT<R>); \
  template __global__ void k_sweep_wave_batch<R, M, PP, true, true, RunOpts>(BatchLaunchT<R>); \
  template __global__ void k_sweep_wave_batch<R, M, PP, false, true, RunOpts>(BatchLaunchT<R>);
#define MHY_SWEEP_WAVE_LAG(R, M) \
  template __global__ void k_sweep_wave_lag<R, M, false, true, RunOpts>(KPT<R>); \
  template __global__ void k_sweep_wave_lag<R, M, false, false, RunOpts>(KPT<R>);
#define MHY_SWEEP_WAVE_INST_R(R) \
  MHY_SWEEP_WAVE_LAG(R, 1) \
  MHY_SWEEP_WAVE_LAG(R, 2) \
  MHY_SWEEP_WAVE_LAG(R, 3) \
  MHY_SWEEP_WAVE_INST(R, 1, false) \
  MHY_SWEEP_WAVE_INST(R, 1, true) \
  MHY_SWEEP_WAVE_INST(R, 2, false) \
  MHY_SWEEP_WAVE_INST(R, 2, true) \
  MHY_SWEEP_WAVE_INST(R, 3, false) \
  MHY_SWEEP_WAVE_INST(R, 3, true)
MHY_SWEEP_WAVE_INST_R(float)

}  // namespace mhy
