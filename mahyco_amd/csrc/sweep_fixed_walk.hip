// Instantiations of the column-walking y sweeps (sweep_walk.hpp): limited slopes
// with their options fixed (FixOpts).
#include "sweep_walk.hpp"

namespace mhy {

// the walkers with their options fixed: sweep 1 with the Lagrange update (0) or after
// the separate Lagrange kernel (1), sweep 2 with the final remap (2)
namespace {
template <class R, int M, int LIM>
SweepFn<R> pickWalk(int sweep) {
  if (sweep == 0) return k_sweep_walk_lag<R, M, FixOpts<LIM, 1>>;
  return sweep == 1 ? k_sweep_walk<R, M, false, FixOpts<LIM, 1>> : k_sweep_walk<R, M, false, FixOpts<LIM, 2>>;
}
}  // namespace
template <class R>
SweepFn<R> sweepFixedWalk(int lim, int m, int sweep) {
  if (!fixedExists(lim, sweep, 0)) return nullptr;
  const bool mm = lim == MHY_LIM_MINMOD;
  if (m == 1) return mm ? pickWalk<R, 1, MHY_LIM_MINMOD>(sweep) : pickWalk<R, 1, MHY_LIM_SUPERBEE>(sweep);
  if (m == 2) return mm ? pickWalk<R, 2, MHY_LIM_MINMOD>(sweep) : pickWalk<R, 2, MHY_LIM_SUPERBEE>(sweep);
  return mm ? pickWalk<R, 3, MHY_LIM_MINMOD>(sweep) : pickWalk<R, 3, MHY_LIM_SUPERBEE>(sweep);
}
template SweepFn<double> sweepFixedWalk<double>(int, int, int);
template SweepFn<float> sweepFixedWalk<float>(int, int, int);

}  // namespace mhy
