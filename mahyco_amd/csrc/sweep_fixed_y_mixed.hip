// Limited-slope wave sweeps along y (mixed form) with their options fixed at compile time
// (FixOpts): minmod and superBee; the fused Lagrange sweep (kind 0), the
// first sweep after the separate Lagrange kernel (1) and the second sweep
// with the final remap (2).
#include "sweep_wave.hpp"

namespace mhy {

namespace {
template <class R, int M, int LIM>
SweepFn<R> pick(int kind) {
  if (kind == 0) return k_sweep_wave_lag<R, M, false, false, FixOpts<LIM, 1>>;
  if (kind == 1) return k_sweep_wave<R, M, false, false, FixOpts<LIM, 1>>;
  return k_sweep_wave<R, M, false, false, FixOpts<LIM, 2>>;
}
template <class R, int M, int LIM>
SweepBatchFn<R> pickBatch(int kind) {
  if (kind == 1) return k_sweep_wave_batch<R, M, false, false, true, FixOpts<LIM, 1>>;
  return k_sweep_wave_batch<R, M, false, false, true, FixOpts<LIM, 2>>;
}
}  // namespace

template <class R>
SweepFn<R> sweepFixedY(int lim, int m, int kind) {
  if (!fixedExists(lim, kind, 0)) return nullptr;
  const bool mm = lim == MHY_LIM_MINMOD;
  if (m == 1) return mm ? pick<R, 1, MHY_LIM_MINMOD>(kind) : pick<R, 1, MHY_LIM_SUPERBEE>(kind);
  if (m == 2) return mm ? pick<R, 2, MHY_LIM_MINMOD>(kind) : pick<R, 2, MHY_LIM_SUPERBEE>(kind);
  return mm ? pick<R, 3, MHY_LIM_MINMOD>(kind) : pick<R, 3, MHY_LIM_SUPERBEE>(kind);
}
template <class R>
SweepBatchFn<R> sweepFixedYBatch(int lim, int m, int kind) {
  if (!fixedExists(lim, kind, 1)) return nullptr;
  const bool mm = lim == MHY_LIM_MINMOD;
  if (m == 1) return mm ? pickBatch<R, 1, MHY_LIM_MINMOD>(kind) : pickBatch<R, 1, MHY_LIM_SUPERBEE>(kind);
  if (m == 2) return mm ? pickBatch<R, 2, MHY_LIM_MINMOD>(kind) : pickBatch<R, 2, MHY_LIM_SUPERBEE>(kind);
  return mm ? pickBatch<R, 3, MHY_LIM_MINMOD>(kind) : pickBatch<R, 3, MHY_LIM_SUPERBEE>(kind);
}
template SweepFn<float> sweepFixedY<float>(int, int, int);
template SweepBatchFn<float> sweepFixedYBatch<float>(int, int, int);

}  // namespace mhy
