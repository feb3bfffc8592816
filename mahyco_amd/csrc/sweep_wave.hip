// Instantiations of the wave-strip sweeps (sweep_wave.hpp): options at run time,
// FP64 form, VNR and Eucclhyd layouts; the launch geometry of every form.
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
MHY_SWEEP_WAVE_INST_R(double)

// the Eucclhyd layouts (FP64 only): momentum (4 + m), and kinetic energy
// (8 + m) for a conservative projection
#define MHY_SWEEP_WAVE_EUC(L)                                          \
  template __global__ void k_sweep_wave<double, L, false, true, RunOpts>(KP);  \
  template __global__ void k_sweep_wave<double, L, false, false, RunOpts>(KP); \
  template __global__ void k_sweep_wave<double, L, true, true, RunOpts>(KP);   \
  template __global__ void k_sweep_wave<double, L, true, false, RunOpts>(KP);
MHY_SWEEP_WAVE_EUC(5)
MHY_SWEEP_WAVE_EUC(6)
MHY_SWEEP_WAVE_EUC(7)
MHY_SWEEP_WAVE_EUC(9)
MHY_SWEEP_WAVE_EUC(10)
MHY_SWEEP_WAVE_EUC(11)
#undef MHY_SWEEP_WAVE_EUC

// threads per block of the wave sweeps: 4 waves along x; along y 4, or 8
// in the mixed form's limited-slope sweeps
unsigned sweepWaveBlock(bool xd, bool mixed, bool pp) {
  return xd ? 256u : 64u * ((mixed && !pp) ? kYWaves<float, false> : kYWaves<double, false>);
}

// launch grid of the wave sweeps (blocks of sweepWaveBlock threads)
dim3 sweepWaveGrid(bool xd, long nx, long ny, bool mixed, bool pp) {
  if (xd) {
    const long strips = (nx + kXOut - 1) / kXOut * ny;
    return dim3((unsigned)((strips + 3) / 4));
  }
  const int W = (mixed && !pp) ? kYWaves<float, false> : kYWaves<double, false>;
  const long gx = (nx + W * kYCols - 1) / (W * kYCols), gy = (ny + kYOut - 1) / kYOut;
  return dim3((unsigned)(gx * gy));
}

}  // namespace mhy
