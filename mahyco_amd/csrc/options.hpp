// Where a kernel's options come from.  RunOpts reads them from the launch
// parameters; FixOpts has them in its type, for the option sets that most runs
// use (second order, a classic limiter, mass-flux dual remap, perfect gases,
// Lagrange + remap without boundary fluxes or periodic cells).  With every
// option a run-time value the sweeps carried all limiters, flux methods and
// both sweep orders through one body: uniform branches that end the
// scheduling regions, scalar work for each, and registers for the union of
// all paths.  Fixed, the one-material FP64 walker of the second sweep shrinks
// from 15.9 to 6.7 KB of code and the two-material PenteBorne x sweep from 58 to
// 15 KB and from 156 to 92 VGPRs (3 to 5 waves per SIMD).  A step, run-time to
// fixed: 200x5 44.5 -> 40.2 us, 256^2 55.8 -> 51.3, 4096^2 2.30 -> 2.13 ms, 500x333
// PenteBorne 103 -> 93 us, 1173x391 three materials 226 -> 189 us, 64-problem mixed
// ensemble 4.55 -> 4.22 ms, Eucclhyd 512^2 180 -> 152 us.  fixedLimiter() is the
// rule that picks the form: it takes exactly the option values the type has,
// every other set runs the run-time form.
#pragma once

#include "common.hpp"

namespace mhy {

struct RunOpts {
  static constexpr int kSweep = 0;  // 1, 2: fixed sweep; 0: either
  static MHY_HD int limiter(const Opts& o) { return o.limiter; }
  static MHY_HD int limiterPure(const Opts& o) { return o.limiter_pure; }
  static MHY_HD int order(const Opts& o) { return o.order; }
  static MHY_HD bool mixte(const Opts& o) { return o.pp_mixte == 1; }
  static MHY_HD bool complet(const Opts& o) { return o.pp_complet == 1; }
  static MHY_HD int methode(const Opts& o) { return o.methode; }
  static MHY_HD bool fluxAny(const Opts& o) { return o.flux_any != 0; }
  static MHY_HD int mode(const Opts& o) { return o.mode; }
  static MHY_HD bool periodic(const Opts& o) { return o.periodic_right != 0; }
  static MHY_HD int eos(const Opts& o, int k) { return o.eos[k]; }
  template <class R>
  static MHY_HD int sweep(const KPT<R>& kp) {
    return kp.sweep;
  }
  template <class R>
  static MHY_HD bool fuse(const KPT<R>& kp) {
    return kp.fuseFinal != 0;
  }
  template <class R>
  static MHY_HD bool geomLoad(const KPT<R>& kp) {
    return kp.geomLoad != 0;
  }
};

// LIM: the limiter (minmod or superBee); SWEEP: first sweep, or second sweep
// with the final remap fused; METHODE: 0 (mass fluxes), or -1 (Eucclhyd: no
// nodal remap); MIXTE, PURE: the PenteBorne-mixte option and its limiter of
// pure cells
template <int LIM, int SWEEP, int METHODE = 0, bool MIXTE = false, int PURE = LIM>
struct FixOpts {
  static constexpr int kSweep = METHODE < 0 ? 1 : SWEEP;  // (Eucclhyd: no fused final remap)
  static MHY_HD int limiter(const Opts&) { return LIM; }
  static MHY_HD int limiterPure(const Opts&) { return PURE; }
  static MHY_HD int order(const Opts&) { return 2; }
  static MHY_HD bool mixte(const Opts&) { return MIXTE; }
  static MHY_HD bool complet(const Opts&) { return false; }
  static MHY_HD int methode(const Opts&) { return METHODE; }
  static MHY_HD bool fluxAny(const Opts&) { return false; }
  static MHY_HD int mode(const Opts&) { return MODE_FULL; }
  static MHY_HD bool periodic(const Opts&) { return false; }
  static MHY_HD int eos(const Opts&, int) { return MHY_EOS_PERFECT_GAS; }
  template <class R>
  static MHY_HD int sweep(const KPT<R>&) {
    return SWEEP;
  }
  template <class R>
  static MHY_HD bool fuse(const KPT<R>&) {
    return SWEEP == 2 && METHODE >= 0;
  }
  template <class R>
  static MHY_HD bool geomLoad(const KPT<R>&) {
    return true;
  }
};

// The limiter of the fixed form these options have, or 0: they run the
// run-time form.  Third order has it too (its own sweeps; the limiter is the
// nodal remap's).
inline int fixedLimiter(const Opts& o) {
  const bool classic = o.limiter == MHY_LIM_MINMOD || o.limiter == MHY_LIM_SUPERBEE;
  bool ok = classic && (o.order == 2 || o.order == 3) && o.mode == MODE_FULL && !o.flux_any && !o.periodic_right &&
            (o.methode == 0 || o.euc) && !(o.pp == 1 && o.pp_complet == 1);
  for (int k = 0; k < o.nbmat; ++k) ok = ok && o.eos[k] == MHY_EOS_PERFECT_GAS;
  return ok ? o.limiter : 0;
}

// The kernels with fixed options exist for these limiters and for the kinds of
// sweep from firstKind on (0: first sweep with the Lagrange update, 1: first sweep, 2: second
// sweep); their pickers return null for anything else.
inline bool fixedExists(int lim, int kind, int firstKind) {
  return (lim == MHY_LIM_MINMOD || lim == MHY_LIM_SUPERBEE) && kind >= firstKind && kind <= 2;
}

}  // namespace mhy
