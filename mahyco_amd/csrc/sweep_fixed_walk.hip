// Instantiations of the column-walking y sweeps (sweep_walk.hpp): limited slopes
// with their options fixed (FixOpts).
#include "sweep_walk.hpp"

namespace mhy {

// the walkers with their options fixed: sweep 1 (after the separate Lagrange
// kernel) or 2 (with the final remap)
namespace {
template <class R, int M, int LIM>
SweepFn<R> pickWalk(int sweep) {
  return sweep == 1 ? k_sweep_walk<R, M, false, FixOpts<LIM, 1>> : k_sweep_walk<R, M, false, FixOpts<LIM, 2>>;
}
}  // namespace
template <class R>
SweepFn<R> sweepFixedWalk(int lim, int m, int sweep) {
  const bool mm = lim == MHY_LIM_MINMOD;
  if (m == 1) return mm ? pickWalk<R, 1, MHY_LIM_MINMOD>(sweep) : pickWalk<R, 1, MHY_LIM_SUPERBEE>(sweep);
  if (m == 2) return mm ? pickWalk<R, 2, MHY_LIM_MINMOD>(sweep) : pickWalk<R, 2, MHY_LIM_SUPERBEE>(sweep);
  return mm ? pickWalk<R, 3, MHY_LIM_MINMOD>(sweep) : pickWalk<R, 3, MHY_LIM_SUPERBEE>(sweep);
}
template SweepFn<double> sweepFixedWalk<double>(int, int, int);
template SweepFn<float> sweepFixedWalk<float>(int, int, int);

}  // namespace mhy
