// Nodal momentum remap of both sweeps in one kernel (remap/DualPhaseRemap1.cc,
// remap/DualPhaseRemap2.cc), after both cell sweeps, for the options the
// fixed sweeps take (second or third order, a classic limiter, mass fluxes).
//
// One sweep at a time the nodal remap is bound by memory: it stores the nodal
// momentum and mass and the Lagrange coordinate of the second axis for the
// next sweep to read back, 8 of the 15 array passes of the pair.  Here a wave
// covers 64 node columns (60 or 59 updated, x or y first; one less with DT) and walks
// down a band of node rows: the
// row-wise sweep works on one node row, its along-x neighbours being the
// adjacent lanes (DPP moves), and the column-wise sweep on the rows the wave
// keeps in registers.  A classic limiter's gradient needs one neighbour on
// each side and an upwind value one gradient on each side, so 2 lanes and 2
// rows at each end are halo.  What goes through memory is read once or
// written once: the Lagrange velocity, the node mass, the mass fluxes of both
// sweeps, and the new velocity.  The Lagrange velocity has a buffer of its own
// (kp.ul, kp.vl): the kernel writes the new one while other waves still read
// the old in their halo.
//
// DT: the new velocity in registers also serves the next step's time step: the wave
// forms the CFL ratio of the cells between its node rows (with the sound speed
// and pressure the second cell sweep has stored) and adds its minimum and the
// maximum pressure to the next step's accumulators, with one node column and one
// row more of halo, instead of the reduction kernel, which reads the velocity back
// and forms the speed of each node four times.
//
// Each dual face is formed once, by the node after it: the mass flux through
// it (the two sides' fluxes are the same sum) and the upwind velocity, which
// the node before takes with a DPP move or from the next row.  The operations
// and operands are those of the one-sweep kernels (remap.hip), so results are
// bitwise the same; the mean over 2 or 4 faces is a product with 1/2 or 1/4.
//
// Measured per step, one kernel per sweep -> this kernel: 256^2 51.3 -> 43.4 us,
// 1531x1021 270 -> 226 us, 4096^2 FP64 2.13 -> 1.81 ms (dual x 0.25 + dual y 0.33 ms
// before), 3072x1024 three materials mixed 780 -> 679 us.
#include <type_traits>

#include "kernels.hpp"
#include "sweep_math.hpp"

namespace mhy {

namespace {

constexpr int kBHalo = 2;
// halo lanes before the updated columns: one more when the column-wise sweep
// comes first, whose result the halo lanes of the row-wise one need and which
// takes the y faces left of a node from the lane before
template <bool XFIRST>
constexpr int kBLeft = XFIRST ? kBHalo : kBHalo + 1;
// node columns updated per wave: with DT the new velocity is also formed one
// column further, for the cells right of the last updated column
template <bool XFIRST, bool DT>
constexpr int kBOut = (DT ? 63 : 64) - kBHalo - kBLeft<XFIRST>;

// value of the lane before / after (the end lanes keep their own)
template <class V>
__device__ __forceinline__ V before(V v) {
  return dppMove<kDppWaveShr1>(v);
}
template <class V>
__device__ __forceinline__ V after(V v) {
  return dppMove<kDppWaveShl1>(v);
}

template <class T>
struct Vel {
  T x, y;
};
// nodal vector of one node: momentum and mass
struct Nodal {
  double x, y, m;
};

// Upwind velocity through the dual face between the node before (pm, gm) and
// this node (p, g): along velocity uN / u0, distance h, mass flux `flux`
// (UtilesDualRemap.cc:234-397; the gradient term times ORD - 1).
template <int ORD, class T>
__device__ __forceinline__ Vel<double> upwindFace(Vel<T> pm, Vel<T> gm, Vel<T> p, Vel<T> g, T uN, T u0, T h, T dtn,
                                                  double flux) {
  const T u = T(0.5) * (uN + u0);
  const int sign = (u > T(0)) ? 1 : -1;
  const T s = T(sign) * h - dtn * u;
  const bool nb = flux > 0;
  const T bx = nb ? pm.x : p.x, by = nb ? pm.y : p.y, gx = nb ? gm.x : g.x, gy = nb ? gm.y : g.y;
  if constexpr (ORD == 2) return {(double)(bx + T(0.5) * gx * s), (double)(by + T(0.5) * gy * s)};
  else return {(double)(bx + T(ORD - 1) * (T(0.5) * gx * s)), (double)(by + T(ORD - 1) * (T(0.5) * gy * s))};
}

// the nodal update from the fluxes through its two faces
__device__ __forceinline__ Nodal updateNode(Nodal u, double minus, double plus, Vel<double> um, Vel<double> up,
                                            bool interior) {
  const Nodal r = {u.x + minus * um.x - plus * up.x, u.y + minus * um.y - plus * up.y, u.m + minus - plus};
  return {interior ? r.x : u.x, interior ? r.y : u.y, interior ? r.m : u.m};
}

template <int LIM, class T>
__device__ __forceinline__ T slope(T gp, T gm) {
  return sw::limitedGradient<T>(LIM, gp, gm, T(0), T(0), T(0), T(0), T(0));
}

}  // namespace

// item: column group and band of this wave (kp.dualRows node rows per band)
template <class R, int M, int LIM, bool XFIRST, bool DT, int ORD>
__device__ __forceinline__ void dualBothBody(const KPT<R>& kp, int item) {
  using T = typename std::conditional<kMixed<R>, float, double>::type;
  const Opts& o = kp.o;
  const auto& f = kp.f;
  const int nx = o.nx, ny = o.ny;
  constexpr int kOut = kBOut<XFIRST, DT>, kLeft = kBLeft<XFIRST>;
  const int groups = (nx + 1 + kOut - 1) / kOut;
  const int rows = kp.dualRows;
  if (item >= groups * ((ny + 1 + rows - 1) / rows)) return;  // the whole wave
  const int lane = threadIdx.x & 63;
  const int t = (item % groups) * kOut - kLeft + lane;
  const int a0 = (item / groups) * rows;
  const int a1 = (a0 + rows - 1 < ny) ? a0 + rows - 1 : ny;
  const bool output = lane >= kLeft && lane < kLeft + kOut && t <= nx;
  const bool intX = t > 0 && t < nx;  // interior along x
  // lanes and rows outside the domain read the nearest node or cell inside:
  // finite values that no updated node uses
  const int tn = t < 0 ? 0 : (t > nx ? nx : t);         // node column
  const int tc = t < 0 ? 0 : (t > nx - 1 ? nx - 1 : t);  // cell column
  const double dtn = f.sc->dt[kp.cur], dt1 = f.sc->dt[kp.nxt];
  const T dtnT = T(dtn);
  // face fluxes along x and along y: those of the sweep in that direction
  double* const* Gx = XFIRST ? f.G : f.G2;
  double* const* Gy = XFIRST ? f.G2 : f.G;
  // means over the faces a dual face touches: 2 per cell row (column)
  const double wy = (t >= 1 && t <= nx - 1) ? 0.25 : 0.5;

  // with DT the walk starts one row early: the cells below the first updated
  // node row belong to this band
  const int first = a0 - kBHalo - (DT ? 1 : 0);

  // what row r of the walk reads: its nodes, the x faces of cell row r and the
  // y faces of row r - 1 (x first), resp. of the rows the updates need
  struct Row {
    R u, v, m;
    double gx[M], gy[M];
  };
  auto load = [&](int r) {
    Row w;
    const int rn = r < 0 ? 0 : (r > ny ? ny : r);
    const long p = (long)rn * (nx + 1) + tn;
    w.u = at(kp.ul, p), w.v = at(kp.vl, p), w.m = at(f.Mp, p);
    const int rx = XFIRST ? r : r - 2;  // cell row of the x faces
    const int rxc = rx < 0 ? 0 : (rx > ny - 1 ? ny - 1 : rx);
    const int ry = r - 1;  // row of the y faces
    const int ryc = ry < 0 ? 0 : (ry > ny ? ny : ry);
#pragma unroll
    for (int k = 0; k < M; ++k) {
      w.gx[k] = at(Gx[k], (long)rxc * (nx + 1) + tn);
      w.gy[k] = at(Gy[k], (long)ryc * nx + tc);
    }
    return w;
  };

  // the walk's state: row r-1 (B) and r-2 (A)
  Vel<T> phA = {T(0), T(0)}, phB = {T(0), T(0)}, gA = {T(0), T(0)}, dB = {T(0), T(0)};
  double ylA = 0.0, ylB = 0.0, fluxA = 0.0;
  Vel<double> upA = {0.0, 0.0};
  Nodal UA = {0.0, 0.0, 0.0}, UB = {0.0, 0.0, 0.0};
  double qx[M], gyP[M];  // x-face pair sums of the cell row before, y faces of the row before
#pragma unroll
  for (int k = 0; k < M; ++k) qx[k] = gyP[k] = 0.0;
  if constexpr (XFIRST) {  // the cell row below the first node row of the walk
    const int c0 = first - 1;
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const double g = at(Gx[k], (long)(c0 < 0 ? 0 : c0) * (nx + 1) + tn);
      qx[k] = g + before(g);
    }
  }

  // mass flux through the x dual face before this node, in the node row
  // between the cell rows of qx and gx; the cell row advances
  auto fluxX = [&](const double* gx, int row) {
    // rows of faces the node touches: cell rows row - 1 and row where they exist
    const bool lo = row >= 1, hi = row <= ny - 1;
    const double w = (lo && hi) ? 0.25 : 0.5;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const double q = gx[k] + before(gx[k]);
      const double p = (lo && hi) ? qx[k] + q : (lo ? qx[k] : q);
      s += p * w;
      qx[k] = q;
    }
    return s;
  };
  // the row-wise sweep of one node row: velocities ph, coordinate xl, flux
  // through the face before each node
  auto sweepX = [&](Vel<T> ph, double xl, Nodal U, double flux) {
    const Vel<T> pm = {before(ph.x), before(ph.y)};
    const double xm = before(xl);
    const T h = T(xl - xm);
    const Vel<T> d = {(ph.x - pm.x) / h, (ph.y - pm.y) / h};
    const Vel<T> dp = {after(d.x), after(d.y)};
    const Vel<T> g = {intX ? slope<LIM>(dp.x, d.x) : T(0), intX ? slope<LIM>(dp.y, d.y) : T(0)};
    const Vel<T> gm = {before(g.x), before(g.y)};
    const Vel<double> um = upwindFace<ORD, T>(pm, gm, ph, g, pm.x, ph.x, h, dtnT, flux);
    const Vel<double> up = {after(um.x), after(um.y)};
    return updateNode(U, flux, after(flux), um, up, intX);
  };

  double vmin = DBL_MAX, pmax = -DBL_MAX, spA = 0.0;
  Row nextRow = load(first);
  for (int r = first; r <= a1 + kBHalo; ++r) {
    const Row w = nextRow;
    if (r < a1 + kBHalo) nextRow = load(r + 1);
    // the cell row between node rows r - 3 and r - 2, for the time step
    double cvol = 0.0, cs = 0.0, pc = 0.0;
    if constexpr (DT) {
      const long cd = (long)(r - 3 < 0 ? 0 : (r - 3 > ny - 1 ? ny - 1 : r - 3)) * nx + tc;
      cvol = at(f.cvol, cd), cs = (double)at(f.c[kp.nxt], cd), pc = (double)at(f.p[kp.nxt], cd);
    }
    const double ux1 = (double)w.u, uy1 = (double)w.v, Mp = (double)w.m;
    Nodal U = {Mp * ux1, Mp * uy1, Mp};
    Vel<T> ph = {T(ux1), T(uy1)};
    const double yl = o.dy * (double)r + uy1 * dt1;
    if constexpr (XFIRST) {
      const double xl = o.dx * (double)t + ux1 * dt1;
      U = sweepX(ph, xl, U, fluxX(w.gx, r));
      ph = {T(U.x / U.m), T(U.y / U.m)};
    }
    // the column-wise sweep: gradient of row B, the face between A and B,
    // update of row A
    const T hN = T(yl - ylB);
    const Vel<T> dN = {(ph.x - phB.x) / hN, (ph.y - phB.y) / hN};
    const bool inB = r - 1 >= 1 && r - 1 <= ny - 1;  // row B has both neighbours
    const Vel<T> gB = {inB ? slope<LIM>(dN.x, dB.x) : T(0), inB ? slope<LIM>(dN.y, dB.y) : T(0)};
    double fluxB = 0.0;  // between rows A and B
#pragma unroll
    for (int k = 0; k < M; ++k) {
      // cell columns t - 1 and t where they exist
      const double c = w.gy[k] + gyP[k], cm = before(c);
      fluxB += ((t >= 1 && t <= nx - 1) ? cm + c : (t >= 1 ? cm : c)) * wy;
      gyP[k] = w.gy[k];
    }
    const Vel<double> upB = upwindFace<ORD, T>(phA, gA, phB, gB, phA.y, phB.y, T(ylB - ylA), dtnT, fluxB);
    const int a = r - 2;
    Nodal V = updateNode(UA, fluxA, fluxB, upA, upB, a >= 1 && a <= ny - 1);
    if constexpr (!XFIRST) {
      // the row-wise second sweep of row A
      const double xl = o.dx * (double)t + (double)phA.x * dt1;
      const Vel<T> p2 = {T(V.x / V.m), T(V.y / V.m)};
      V = sweepX(p2, xl, V, fluxX(w.gx, a));
    }
    // remapVariables, nodes (PhaseRemapFinal.cc:207-234)
    const R vx = (R)(V.x / V.m), vy = (R)(V.y / V.m);
    if (output && a >= a0 && a <= a1) {
      const long p = (long)a * (nx + 1) + t;
      at(f.ux[kp.nxt], p) = vx;
      at(f.uy[kp.nxt], p) = vy;
    }
    if constexpr (DT) {
      // computeDeltaT (VnrRemap.cc:14-50) of the cell between node rows a-1 and
      // a, in the reduction kernel's order of the four nodes
      const double wx = (double)vx, wv = (double)vy;
      const double sp = sqrt(wx * wx + wv * wv) * 0.25;
      const double spAr = after(spA), spr = after(sp);
      if (output && t < nx && a >= 1 && a >= a0 && a <= a1) {
        const double uc = ((0.0 + spA + spAr) + spr) + sp;
        vmin = smin(vmin, cvol / (o.cfl_euler * uc + cs));
        pmax = (pc > pmax) ? pc : pmax;
      }
      spA = sp;
    }
    phA = phB, phB = ph, gA = gB, dB = dN;
    ylA = ylB, ylB = yl, fluxA = fluxB, upA = upB;
    UA = UB, UB = U;
  }
  // the wave's extrema into the next step's accumulators (a slot that already
  // holds a better value is left alone: it only improves)
  if constexpr (!DT) return;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    vmin = smin(vmin, __shfl_xor(vmin, off, 64));
    const double v = __shfl_xor(pmax, off, 64);
    pmax = (v > pmax) ? v : pmax;
  }
  if (lane == 0) {
    unsigned long long* slot = f.keys->k[kp.nxt][item % kDtSlots];
    const unsigned long long lo = dkeyPos(vmin), hi = dkeySigned(pmax);
    if (lo < __hip_atomic_load(&slot[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&slot[0], lo);
    if (hi > __hip_atomic_load(&slot[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&slot[1], hi);
  }
}

// (a wave past the last band leaves at once: the kernel has no barrier)
template <class R, int M, int LIM, bool XFIRST, bool DT, int ORD>
__global__ __launch_bounds__(256) void k_dual_both(KPT<R> kp) {
  dualBothBody<R, M, LIM, XFIRST, DT, ORD>(kp, (int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
}
// all problems of an ensemble in one launch, one workgroup per virtual block
template <class R, int M, int LIM, bool XFIRST, bool DT, int ORD>
__global__ __launch_bounds__(256) void k_dual_both_batch(BatchLaunchT<R> bl) {
  batchRun<true>(bl, [&](const KPT<R>& kp, unsigned local, unsigned, unsigned) {
    dualBothBody<R, M, LIM, XFIRST, DT, ORD>(kp, (int)(local * 4 + (threadIdx.x >> 6)));
  });
}

// The next step's CFL reduction rides along in bands of at least 16 rows, where
// its extra halo row is cheap (us per step, in the kernel / as a kernel of its own:
// 4096^2 1790 / 1809, 1531x1021 220 / 226); a mesh of shorter bands is bound by the
// length of the walk, and the reduction kernel overlaps nothing but takes less
// than the longer walk (256^2 45.5 / 43.4, 1173x391 164 / 159).
bool dualBothDt(int rows) { return rows >= 16; }

int dualBothItems(long nx, long ny, int rows, bool xfirst) {
  const long out = dualBothDt(rows) ? (xfirst ? kBOut<true, true> : kBOut<false, true>)
                                    : (xfirst ? kBOut<true, false> : kBOut<false, false>);
  return (int)((nx + 1 + out - 1) / out * ((ny + 1 + rows - 1) / rows));
}

// Node rows per band, from the number of waves each choice leaves: a band has 4
// halo rows, but a wave walks its band row after row, so a mesh that cannot fill
// the chip wants more, shorter bands.  32 rows where that leaves a wave for each
// of the 4096 wave slots (4 per SIMD), else the longest band that leaves about
// 0.7 waves per SIMD.  us per step, by rows: 200x5 (12 waves at 2 rows) 2: 36.6, 4: 38.7;
// 256^2 2: 43.4, 4: 45.3, 16: 58.5; 500x333 PenteBorne 2: 78.6, 4: 77.3, 8: 82.5;
// 1173x391 three materials 4: 160.0, 8: 158.6, 16: 169.0; 1531x1021 8: 228, 16: 226,
// 32: 233; 2048^2 mixed 8: 455, 16: 443, 32: 456; 4096^2 16: 1824, 32: 1809, 64: 1829.
int dualBothRows(long waves2) {
  // (waves2: waves at 2 rows per band; they halve with each doubling)
  if (waves2 / 16 >= 4096) return 32;
  int rows = 16;
  while (rows > 2 && waves2 / (rows / 2) < 700) rows /= 2;
  return rows;
}

namespace {
template <class R, int M, int LIM, int ORD>
SweepFn<R> pick(bool xfirst, bool dt) {
  if (dt) return xfirst ? k_dual_both<R, M, LIM, true, true, ORD> : k_dual_both<R, M, LIM, false, true, ORD>;
  return xfirst ? k_dual_both<R, M, LIM, true, false, ORD> : k_dual_both<R, M, LIM, false, false, ORD>;
}
template <class R, int M, int LIM>
SweepBatchFn<R> pickBatch(bool xfirst, bool dt) {
  if (dt) return xfirst ? k_dual_both_batch<R, M, LIM, true, true, 2> : k_dual_both_batch<R, M, LIM, false, true, 2>;
  return xfirst ? k_dual_both_batch<R, M, LIM, true, false, 2> : k_dual_both_batch<R, M, LIM, false, false, 2>;
}
template <class R, int M>
SweepFn<R> pickLim(int lim, bool xf, bool dt, int order) {
  if (order == 3)
    return lim == MHY_LIM_MINMOD ? pick<R, M, MHY_LIM_MINMOD, 3>(xf, dt) : pick<R, M, MHY_LIM_SUPERBEE, 3>(xf, dt);
  return lim == MHY_LIM_MINMOD ? pick<R, M, MHY_LIM_MINMOD, 2>(xf, dt) : pick<R, M, MHY_LIM_SUPERBEE, 2>(xf, dt);
}
}  // namespace
template <class R>
SweepFn<R> dualBothKernel(int lim, int m, bool xf, int rows, int order) {
  if (!fixedExists(lim, 1, 1)) return nullptr;
  const bool dt = dualBothDt(rows);
  return m == 1 ? pickLim<R, 1>(lim, xf, dt, order) : m == 2 ? pickLim<R, 2>(lim, xf, dt, order) : pickLim<R, 3>(lim, xf, dt, order);
}
template <class R>
SweepBatchFn<R> dualBothBatchKernel(int lim, int m, bool xf, int rows) {
  if (!fixedExists(lim, 1, 1)) return nullptr;
  const bool dt = dualBothDt(rows);
  const bool mm = lim == MHY_LIM_MINMOD;
  if (m == 1) return mm ? pickBatch<R, 1, MHY_LIM_MINMOD>(xf, dt) : pickBatch<R, 1, MHY_LIM_SUPERBEE>(xf, dt);
  if (m == 2) return mm ? pickBatch<R, 2, MHY_LIM_MINMOD>(xf, dt) : pickBatch<R, 2, MHY_LIM_SUPERBEE>(xf, dt);
  return mm ? pickBatch<R, 3, MHY_LIM_MINMOD>(xf, dt) : pickBatch<R, 3, MHY_LIM_SUPERBEE>(xf, dt);
}
template SweepFn<double> dualBothKernel<double>(int, int, bool, int, int);
template SweepFn<float> dualBothKernel<float>(int, int, bool, int, int);
template SweepBatchFn<double> dualBothBatchKernel<double>(int, int, bool, int);
template SweepBatchFn<float> dualBothBatchKernel<float>(int, int, bool, int);

}  // namespace mhy
