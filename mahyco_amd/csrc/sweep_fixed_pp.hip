// PenteBorne wave sweeps (FP64) with their options fixed at compile time
// (FixOpts): minmod and superBee, VNR without the mixte option, and the
// Eucclhyd layouts of a non-conservative projection with and without it
// (pure-cell limiter arithmeticG).
#include "sweep_wave.hpp"

namespace mhy {

namespace {
template <int M, bool XD, int LIM>
SweepFn<double> pickPP(int sweep) {
  if constexpr (XD) {
    if (sweep == 0) return k_sweep_wave_lag<double, M, true, XD, FixOpts<LIM, 1>>;
  }
  if (sweep == 1) return k_sweep_wave<double, M, true, XD, FixOpts<LIM, 1>>;
  return k_sweep_wave<double, M, true, XD, FixOpts<LIM, 2>>;
}
template <int M, bool XD>
SweepFn<double> pickPPLim(int lim, int sweep) {
  return lim == MHY_LIM_MINMOD ? pickPP<M, XD, MHY_LIM_MINMOD>(sweep) : pickPP<M, XD, MHY_LIM_SUPERBEE>(sweep);
}
template <int L, bool XD, bool MIXTE>
SweepFn<double> pickEuc(int sweep) {
  constexpr int pure = MIXTE ? MHY_LIM_ARITHMETICG : MHY_LIM_SUPERBEE;
  if (sweep == 1) return k_sweep_wave<double, L, true, XD, FixOpts<MHY_LIM_SUPERBEE, 1, -1, MIXTE, pure>>;
  return k_sweep_wave<double, L, true, XD, FixOpts<MHY_LIM_SUPERBEE, 2, -1, MIXTE, pure>>;
}
template <int L>
SweepFn<double> pickEucDir(bool xd, bool mixte, int sweep) {
  if (mixte) return xd ? pickEuc<L, true, true>(sweep) : pickEuc<L, false, true>(sweep);
  return xd ? pickEuc<L, true, false>(sweep) : pickEuc<L, false, false>(sweep);
}
}  // namespace

SweepFn<double> sweepFixedPP(bool xd, int lim, int m, int sweep) {
  if (!fixedExists(lim, sweep, xd ? 0 : 1)) return nullptr;
  if (m == 1) return xd ? pickPPLim<1, true>(lim, sweep) : pickPPLim<1, false>(lim, sweep);
  if (m == 2) return xd ? pickPPLim<2, true>(lim, sweep) : pickPPLim<2, false>(lim, sweep);
  return xd ? pickPPLim<3, true>(lim, sweep) : pickPPLim<3, false>(lim, sweep);
}

// superBee
SweepFn<double> sweepFixedEuc(bool xd, int m, bool mixte, int sweep) {
  if (!fixedExists(MHY_LIM_SUPERBEE, sweep, 1)) return nullptr;
  if (m == 1) return pickEucDir<5>(xd, mixte, sweep);
  if (m == 2) return pickEucDir<6>(xd, mixte, sweep);
  return pickEucDir<7>(xd, mixte, sweep);
}

}  // namespace mhy
