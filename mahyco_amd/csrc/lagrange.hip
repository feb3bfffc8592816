// Lagrange phase of the VNR scheme on CDNA4: CFL time-step / max-pressure
// reduction, nodal momentum update with boundary conditions, and the cell
// update (sub-volumes, densities, artificial viscosity, energy, perfect-gas
// EOS) fused with the preparation of the remap vectors.
//
// Arithmetic follows the reference operation by operation (compiled with
// -ffp-contract=off), so FP64 results are bitwise those of the CPU path.
#include "common.hpp"
#include "kernels.hpp"
#include "lagrange_cell.hpp"

namespace mhy {

namespace {

__device__ __forceinline__ double waveMin(double v) {
  for (int o = 32; o > 0; o >>= 1) v = smin(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ double waveMax(double v) {
  for (int o = 32; o > 0; o >>= 1) {
    double w = __shfl_xor(v, o, 64);
    v = (w > v) ? w : v;
  }
  return v;
}

// node coordinates at the step start
template <class R>
__device__ __forceinline__ D2 nodeX(const KPT<R>& kp, long j, long i) {
  if (kp.o.mode == MODE_LAGRANGE) {
    long p = j * (kp.o.nx + 1) + i;
    return {kp.f.X[kp.cur][p], kp.f.Y[kp.cur][p]};
  }
  return eulerNode(kp.o, j, i);
}

}  // namespace

// vnr_remap/VnrRemap.cc:14-50 (computeDeltaT) fused with the max-pressure
// reduction of PhaseLagrange.cc:55-61.  Min and max ignore NaN values like
// the reference's reducers.  Each block reduces its cells and adds them to
// the step's accumulators with one 64-bit atomic min / max (exact and
// order-free, no fence); the node update then forms dt and t (computeTime).
// b: block index among the nb blocks working on this problem.  The
// reduction is FP64 in both forms (FP32 inputs are widened).
template <class R>
__device__ __forceinline__ void dtReduceBody(const KPT<R>& kp, unsigned b, unsigned nb) {
  const Opts& o = kp.o;
  const auto& f = kp.f;
  const long nx = o.nx;
  double vmin = DBL_MAX, pm = -DBL_MAX;
  const R* ux = f.ux[kp.cur];
  const R* uy = f.uy[kp.cur];
  for (long c = (long)b * blockDim.x + threadIdx.x; c < kp.ncell; c += (long)nb * blockDim.x) {
    // 32-bit division: cell and node counts stay below 2^31 (checked at set-up)
    const long j = (long)((unsigned)c / (unsigned)nx), i = c - j * nx;
    const long p0 = j * (nx + 1) + i;
    const long nd[4] = {p0, p0 + 1, p0 + nx + 2, p0 + nx + 1};
    double uc = 0.0;
    for (int s = 0; s < 4; ++s) {
      const double a = ux[nd[s]], b = uy[nd[s]];
      uc += sqrt(a * a + b * b) * 0.25;
    }
    // (the numerator of the fixed cells is formed once, at set-up)
    const double cv = f.cvol ? f.cvol[c] : o.cfl * sqrt(f.vol[kp.cur][c]);
    const double v = cv / (o.cfl_euler * uc + (double)f.c[kp.cur][c]);
    vmin = smin(vmin, v);
    const double pc = f.p[kp.cur][c];
    pm = (pc > pm) ? pc : pm;
  }
  __shared__ double smn[4], smx[4];
  vmin = waveMin(vmin);
  pm = waveMax(pm);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) smn[w] = vmin, smx[w] = pm;
  __syncthreads();
  if (threadIdx.x == 0) {
    double lo = smn[0], hi = smx[0];
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) lo = smin(lo, smn[k]), hi = (smx[k] > hi) ? smx[k] : hi;
    unsigned long long* slot = f.keys->k[kp.cur][b % kDtSlots];
    atomicMin(&slot[0], dkeyPos(lo));
    atomicMax(&slot[1], dkeySigned(hi));
  }
}

template <class R>
__global__ __launch_bounds__(256) void k_dt_reduce(KPT<R> kp) {
  dtReduceBody(kp, blockIdx.x, gridDim.x);
}

// dt_{n+1} = min(CFL minimum, 1.05 dt_n) (VnrRemap.cc:45-50) and the maximum
// pressure, from the step's accumulators (the same value for every thread
// that folds them).
struct DtNow {
  double dt1, pmax;
};
template <class R>
__device__ __forceinline__ DtNow dtFold(const FieldsT<R>& f, int cur) {
  unsigned long long lo = f.keys->k[cur][0][0], hi = f.keys->k[cur][0][1];
#pragma unroll
  for (int s = 1; s < kDtSlots; ++s) {
    const unsigned long long a = f.keys->k[cur][s][0], b = f.keys->k[cur][s][1];
    lo = (a < lo) ? a : lo;
    hi = (b > hi) ? b : hi;
  }
  return {smin(dkeyPosInv(lo), 1.05 * f.sc->dt[cur]), dkeySignedInv(hi)};
}
// stores dt_{n+1}, t_{n+1} (computeTime) and the maximum pressure and resets
// the accumulators of the next step's parity (one thread)
template <class R>
__device__ __forceinline__ void dtStore(const FieldsT<R>& f, int cur, int nxt, DtNow d) {
  Scalars* sc = f.sc;
  sc->dt[nxt] = d.dt1;
  sc->t[nxt] = sc->t[cur] + d.dt1;
  sc->pmax = d.pmax;
#pragma unroll
  for (int s = 0; s < kDtSlots; ++s) {
    f.keys->k[nxt][s][0] = dkeyPos(DBL_MAX);
    f.keys->k[nxt][s][1] = dkeySigned(-DBL_MAX);
  }
}
// dt_{n+1} for the node update; first: the one thread that stores it.  The
// step's other kernels come later and read the stored value.
template <class R>
__device__ __forceinline__ double dtForNodes(const KPT<R>& kp, bool first) {
  if (!kp.dtFold) return kp.f.sc->dt[kp.nxt];
  const DtNow d = dtFold(kp.f, kp.cur);
  if (first) dtStore(kp.f, kp.cur, kp.nxt, d);
  return d.dt1;
}

// cfl sqrt(vol) of the fixed Euler cells (set-up)
template <class R>
__global__ __launch_bounds__(256) void k_cfl_volume(KPT<R> kp) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < kp.ncell) kp.f.cvol[c] = kp.o.cfl * sqrt(kp.f.vol[0][c]);
}
// empties the accumulators of the current parity
template <class R>
__global__ void k_dt_reset(KPT<R> kp) {
  if (threadIdx.x < kDtSlots && blockIdx.x == 0) {
    kp.f.keys->k[kp.cur][threadIdx.x][0] = dkeyPos(DBL_MAX);
    kp.f.keys->k[kp.cur][threadIdx.x][1] = dkeySigned(-DBL_MAX);
  }
}

template <class R>
__global__ void k_dt_finalize(KPT<R> kp) {
  if (threadIdx.x == 0 && blockIdx.x == 0) dtStore(kp.f, kp.cur, kp.nxt, dtFold(kp.f, kp.cur));
}

// sansLagrange: deltat_nplus1 = deltat_n (VnrRemap.cc:143-146)
template <class R>
__global__ void k_dt_hold(KPT<R> kp) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    Scalars* sc = kp.f.sc;
    sc->dt[kp.nxt] = sc->dt[kp.cur];
    sc->t[kp.nxt] = sc->t[kp.cur] + sc->dt[kp.nxt];
  }
}

// Node kernel: node mass as the mean of the adjacent cell masses
// (PhaseLagrange.cc:31-48), then updateVelocity (PhaseLagrange.cc:167-197),
// updateVelocityBoundaryConditions (ConditionsLimites.cc:12-185) and
// updatePosition (PhaseLagrange.cc:203-208).  In advection mode the velocity
// is carried over unchanged (VnrRemap.cc:152-154).  Arithmetic is FP64 in
// both forms.
template <class R>
__device__ __forceinline__ void lagrangeNodeAt(const KPT<R>& kp, double dt1, long p, long j, long i) {
  const Opts& o = kp.o;
  const auto& f = kp.f;
  const long nx = o.nx, ny = o.ny;
  // cells of the node in getCellsOfNode order (CartesianMesh2D.cc:97-108)
  const bool hc[4] = {j < ny && i < nx, j < ny && i > 0, j > 0 && i < nx, j > 0 && i > 0};
  // a missing cell reads the existing one nearest to it and is left out of the
  // sums: the loads of the four wait for no branch.  The boundary nodes set
  // the length of the node update on the smallest meshes (200x5: a pass of 50
  // steps 1920 -> 1843 us; 256x256 and larger unchanged)
  const long jl = j > 0 ? j - 1 : 0, jh = j < ny ? j : ny - 1, il = i > 0 ? i - 1 : 0, ih = i < nx ? i : nx - 1;
  const long cc[4] = {jh * nx + ih, jh * nx + il, jl * nx + ih, jl * nx + il};
  double mq[4], pq[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    mq[q] = f.M[cc[q]];
    pq[q] = (double)f.p[kp.cur][cc[q]] + (double)f.q[kp.cur][cc[q]];
  }
  double msum = 0.0;
  int cnt = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    msum = hc[q] ? msum + mq[q] : msum;
    cnt += hc[q] ? 1 : 0;
  }
  const double Mp = msum / (double)cnt;
  f.Mp[p] = Mp;
  const double uxn = (double)f.ux[kp.cur][p], uyn = (double)f.uy[kp.cur][p];
  if (o.mode == MODE_ADVECTION) {
    kp.ul[p] = uxn;
    kp.vl[p] = uyn;
    return;
  }
  const double dt = 0.5 * (dt1 + f.sc->dt[kp.cur]);
  // corner normals of the four cells at this node: C(cell, node) depends on
  // the node and its two neighbours along the cell's edges
  const D2 X0 = nodeX(kp, j, i);
  D2 Cn[4];
  if (o.mode == MODE_LAGRANGE) {
    if (hc[0]) Cn[0] = lpcNpc(X0, nodeX(kp, j, i + 1), nodeX(kp, j + 1, i));
    if (hc[1]) Cn[1] = lpcNpc(X0, nodeX(kp, j + 1, i), nodeX(kp, j, i - 1));
    if (hc[2]) Cn[2] = lpcNpc(X0, nodeX(kp, j - 1, i), nodeX(kp, j, i + 1));
    if (hc[3]) Cn[3] = lpcNpc(X0, nodeX(kp, j, i - 1), nodeX(kp, j - 1, i));
  } else {  // fixed Euler grid: axis-aligned edges
    Cn[0] = lpcNpcAxis(X0, eulerNode(o, j, i + 1), eulerNode(o, j + 1, i));
    Cn[1] = lpcNpcAxis(X0, eulerNode(o, j + 1, i), eulerNode(o, j, i - 1));
    Cn[2] = lpcNpcAxis(X0, eulerNode(o, j - 1, i), eulerNode(o, j, i + 1));
    Cn[3] = lpcNpcAxis(X0, eulerNode(o, j, i - 1), eulerNode(o, j - 1, i));
  }
  const bool inner = (i != 0 && j != 0 && i != nx && j != ny);
  D2 un = {uxn, uyn};
  D2 u1;
  if (inner) {
    D2 r = {0.0, 0.0};
    for (int q = 0; q < 4; ++q) r = d2add(r, d2mul(Cn[q], pq[q]));
    u1 = d2add(un, d2mul(r, dt / Mp));
    if (o.mode == MODE_LAGRANGE) f.outvx[p] = u1.x, f.outvy[p] = u1.y;
  } else {
    // sides in the reference's launch order, then corners; a side that is
    // neither symmetry nor imposed velocity leaves the buffer unchanged
    u1 = {(double)f.ux[kp.nxt][p], (double)f.uy[kp.nxt][p]};
    auto side = [&](int bc, D2 axis, const double* val) {
      if (bc == MHY_BC_SYMMETRY) {
        D2 r = {0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const D2 s = d2add(r, d2mul(d2add(Cn[q], symmetricVector(Cn[q], axis)), pq[q]));
          r = {hc[q] ? s.x : r.x, hc[q] ? s.y : r.y};
        }
        u1 = d2add(un, d2mul(r, dt / (Mp)));
      } else if (bc == MHY_BC_IMPOSED_VELOCITY) {
        u1 = {val[0], val[1]};
      }
    };
    const D2 ax = {1.0, 0.0}, ay = {0.0, 1.0};
    if (j == 0) side(o.bc_bottom, ax, o.bcv_bottom);
    if (j == ny) side(o.bc_top, ax, o.bcv_top);
    if (i == 0) side(o.bc_left, ay, o.bcv_left);
    if (i == nx) side(o.bc_right, ay, o.bcv_right);
    auto corner = [&](int a, int b, const double* val) {
      if (a == MHY_BC_SYMMETRY && b == MHY_BC_SYMMETRY) u1 = {0.0, 0.0};
      else if (a == MHY_BC_IMPOSED_VELOCITY && b == MHY_BC_IMPOSED_VELOCITY) u1 = {val[0], val[1]};
    };
    if (j == ny && i == 0) corner(o.bc_top, o.bc_left, o.bcv_left);
    if (j == ny && i == nx) corner(o.bc_top, o.bc_right, o.bcv_right);
    if (j == 0 && i == 0) corner(o.bc_bottom, o.bc_left, o.bcv_left);
    if (j == 0 && i == nx) corner(o.bc_bottom, o.bc_right, o.bcv_right);
  }
  kp.ul[p] = u1.x;
  kp.vl[p] = u1.y;
  if (o.mode == MODE_LAGRANGE) {
    f.X[kp.nxt][p] = X0.x + u1.x * dt1;
    f.Y[kp.nxt][p] = X0.y + u1.y * dt1;
  }
}

// One thread per node, any mode (b: block index inside the problem).
template <class R>
__device__ __forceinline__ void lagrangeNodeBody(const KPT<R>& kp, unsigned b) {
  const double dt1 = dtForNodes(kp, b == 0 && threadIdx.x == 0);
  const long p = (long)b * blockDim.x + threadIdx.x;
  if (p >= kp.nnode) return;
  const long nx = kp.o.nx;
  const long j = (long)((unsigned)p / (unsigned)(nx + 1)), i = p - j * (nx + 1);
  lagrangeNodeAt(kp, dt1, p, j, i);
}

template <class R>
__global__ __launch_bounds__(256) void k_lagrange_node(KPT<R> kp) {
  lagrangeNodeBody(kp, blockIdx.x);
}

// The node update on the fixed Euler grid (MODE_FULL).  A wave takes 64 interior
// node columns and walks up a band of kp.nodeRows node rows: each row's cell
// masses and pressures are read once and serve the node rows below and above
// it; the waves after the last band take 64 boundary nodes each (bottom row,
// top row, then the left and right columns without their corners) through the
// general body with its conditions.  Interior nodes have four cells, and the
// corner normals are the raw half-edge sums; operands and order are those of
// lagrangeNodeAt, so the results are bitwise its own.
//
// Bound by memory on large meshes (8 array passes in FP64) and by the latency of
// the chain keys -> dt -> update on small ones; the cell loads come before the
// fold so that the two overlap.  One launch does the whole of it: a finalize
// kernel (2 to 5 us) and a boundary-node kernel (5 to 7 us) of their own cost
// 4.9 us of a 256^2 step; one thread per interior node reading its four cells took
// 27 us on 1531x1021 cells and 244 us in the 64-problem mixed ensemble, whose steps
// went from 220 to 215 us and from 2945 to 2855 us.
template <class R>
__device__ __forceinline__ void lagrangeNodeWalk(const KPT<R>& kp, int item) {
  const Opts& o = kp.o;
  const auto& f = kp.f;
  const int nx = o.nx, ny = o.ny, rows = kp.nodeRows;
  const int lane = threadIdx.x & 63;
  const int groups = (nx - 1 + 63) / 64, bands = (ny - 1 + rows - 1) / rows;
  const bool first = (item == 0 && lane == 0);
  if (item >= groups * bands) {
    const int e = (item - groups * bands) * 64 + lane;
    const double dt1 = dtForNodes(kp, first);
    int j, i;
    if (e < nx + 1) {
      j = 0, i = e;
    } else if (e < 2 * (nx + 1)) {
      j = ny, i = e - (nx + 1);
    } else if (e < 2 * (nx + 1) + (ny - 1)) {
      j = 1 + (e - 2 * (nx + 1)), i = 0;
    } else if (e < 2 * (nx + 1) + 2 * (ny - 1)) {
      j = 1 + (e - 2 * (nx + 1) - (ny - 1)), i = nx;
    } else {
      return;
    }
    lagrangeNodeAt(kp, dt1, (long)j * (nx + 1) + i, j, i);
    return;
  }
  const int i = 1 + (item % groups) * 64 + lane;
  const int ic = i < nx ? i : nx - 1;  // lanes past the last column repeat it
  const int j0 = 1 + (item / groups) * rows;
  const int j1 = (j0 + rows - 1 < ny - 1) ? j0 + rows - 1 : ny - 1;
  // cells (j, i) and (j, i-1) of a row: mass and pressure + pseudo
  struct Cells {
    double m0, m1, p0, p1;
  };
  auto loadCells = [&](int j) {
    const int c = j * nx + ic;
    Cells w;
    w.m0 = at(f.M, c), w.m1 = at(f.M - 1, c);
    w.p0 = (double)at(f.p[kp.cur], c) + (double)at(f.q[kp.cur], c);
    w.p1 = (double)at(f.p[kp.cur] - 1, c) + (double)at(f.q[kp.cur] - 1, c);
    return w;
  };
  Cells lo = loadCells(j0 - 1), hi = loadCells(j0);
  const double dt1 = dtForNodes(kp, first);
  const double dt = 0.5 * (dt1 + f.sc->dt[kp.cur]);
  for (int j = j0; j <= j1; ++j) {
    const int p = j * (nx + 1) + ic;
    const double uxn = (double)at(f.ux[kp.cur], p), uyn = (double)at(f.uy[kp.cur], p);
    const Cells next = (j < j1) ? loadCells(j + 1) : hi;
    const double Mp = ((((0.0 + hi.m0) + hi.m1) + lo.m0) + lo.m1) / 4.0;
    const D2 X0 = eulerNode(o, j, ic);
    const D2 Cn[4] = {lpcNpcAxis(X0, eulerNode(o, j, ic + 1), eulerNode(o, j + 1, ic)),
                      lpcNpcAxis(X0, eulerNode(o, j + 1, ic), eulerNode(o, j, ic - 1)),
                      lpcNpcAxis(X0, eulerNode(o, j - 1, ic), eulerNode(o, j, ic + 1)),
                      lpcNpcAxis(X0, eulerNode(o, j, ic - 1), eulerNode(o, j - 1, ic))};
    D2 r = {0.0, 0.0};
    r = d2add(r, d2mul(Cn[0], hi.p0));
    r = d2add(r, d2mul(Cn[1], hi.p1));
    r = d2add(r, d2mul(Cn[2], lo.p0));
    r = d2add(r, d2mul(Cn[3], lo.p1));
    const D2 u1 = d2add(D2{uxn, uyn}, d2mul(r, dt / Mp));
    if (i < nx) {
      at(f.Mp, p) = Mp;
      at(kp.ul, p) = u1.x;
      at(kp.vl, p) = u1.y;
    }
    lo = hi, hi = next;
  }
}

template <class R>
__global__ __launch_bounds__(256) void k_lagrange_node_walk(KPT<R> kp) {
  const int item = (int)(blockIdx.x * 4) + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  lagrangeNodeWalk(kp, item);
}

// waves of the kernel: bands of interior nodes, then 64 boundary nodes each
int nodeWalkItems(long nx, long ny, int rows) {
  const long nedge = 2 * (nx + 1) + 2 * (ny - 1);
  return (int)((nx - 1 + 63) / 64 * ((ny - 1 + rows - 1) / rows) + (nedge + 63) / 64);
}

// Node rows per band, from the waves that one row each leaves: 4 rows where that
// still leaves 512, else one.  us per step by rows: 256^2 (1020 waves) 1: 42.4, 4:
// 42.6; 500x333 PenteBorne 1: 76.3, 4: 75.5; 1173x391 1: 161.5, 2: 157.8, 4: 158.7;
// 1531x1021 1: 221, 4: 215, 8: 216; 2048^2 mixed 1: 450, 2: 432, 4: 435, 16: 436; 4096^2
// 1: 1831, 4: 1764, 16: 1797; 64-problem mixed ensemble 1: 2957, 4: 2860, 8: 2853.
int nodeWalkRows(long waves1) { return waves1 >= 2048 ? 4 : 1; }

// Cell kernel: the cell part of the Lagrange phase (lagrangeCellCompute,
// lagrange_cell.hpp) with the remap vector, the Lagrange volume and centroid
// (and the Lagrange density / pseudo where the options need them) stored for
// the first remap sweep.  The wave sweeps fuse this update into their first
// sweep instead; this kernel serves the other sweep kernels and the
// moving-mesh mode.
template <class R, int M>
__device__ __forceinline__ void lagrangeCellBody(const KPT<R>& kp, unsigned b) {
  const long c = (long)b * blockDim.x + threadIdx.x;
  if (c >= kp.ncell) return;
  const long nx = kp.o.nx;
  const long j = (long)((unsigned)c / (unsigned)nx), i = c - j * nx;
  LagCell<M> lc;
  if (!lagrangeCellCompute<R, M>(kp, c, j, i, true, lc)) return;
  const auto& f = kp.f;
#pragma unroll
  for (int q = 0; q < 3 * M + 1; ++q) at(f.UL[q], c) = lc.U[q];
  at(f.VL, c) = lc.V;
  if (kp.o.methode == 1) at(f.rL, c) = lc.rho;
  if (kp.o.pp == 1) at(f.qL, c) = lc.q;
  at(f.XcL, c) = lc.xc.x;
  at(f.YcL, c) = lc.xc.y;
}

template <class R, int M>
__global__ __launch_bounds__(256) void k_lagrange_cell(KPT<R> kp) {
  lagrangeCellBody<R, M>(kp, blockIdx.x);
}

// ---------------------------------------------------------------- batches
// One launch serves every problem of an ensemble: the virtual blocks of all
// problems are numbered consecutively (BatchLaunch::start) and a fixed
// number of workgroups walks them.

template <class R, bool ONE>
__global__ __launch_bounds__(256) void k_dt_reduce_batch(BatchLaunchT<R> bl) {
  batchRun<ONE>(bl, [&](const KPT<R>& kp, unsigned b, unsigned, unsigned nb) {
    dtReduceBody(kp, b, nb);
    __syncthreads();  // the shared scratch is reused by the next virtual block
  });
}
template <class R>
__global__ __launch_bounds__(256) void k_lagrange_node_batch(BatchLaunchT<R> bl) {
  batchRun<true>(bl, [&](const KPT<R>& kp, unsigned local, unsigned, unsigned) {
    lagrangeNodeWalk(kp, (int)(local * 4) + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)));
  });
}
template <class R, int M, bool ONE>
__global__ __launch_bounds__(256) void k_lagrange_cell_batch(BatchLaunchT<R> bl) {
  batchRun<ONE>(bl, [&](const KPT<R>& kp, unsigned b, unsigned, unsigned) { lagrangeCellBody<R, M>(kp, b); });
}

#define MHY_LAGRANGE_INST_ONE(R, ONE)                                        \
  template __global__ void k_dt_reduce_batch<R, ONE>(BatchLaunchT<R>);       \
  template __global__ void k_lagrange_cell_batch<R, 1, ONE>(BatchLaunchT<R>); \
  template __global__ void k_lagrange_cell_batch<R, 2, ONE>(BatchLaunchT<R>); \
  template __global__ void k_lagrange_cell_batch<R, 3, ONE>(BatchLaunchT<R>);
#define MHY_LAGRANGE_INST(R)                                                 \
  template __global__ void k_dt_reduce<R>(KPT<R>);                           \
  template __global__ void k_dt_finalize<R>(KPT<R>);                         \
  template __global__ void k_cfl_volume<R>(KPT<R>);                          \
  template __global__ void k_dt_reset<R>(KPT<R>);                            \
  template __global__ void k_dt_hold<R>(KPT<R>);                             \
  template __global__ void k_lagrange_node<R>(KPT<R>);                       \
  template __global__ void k_lagrange_node_walk<R>(KPT<R>);                  \
  template __global__ void k_lagrange_node_batch<R>(BatchLaunchT<R>);        \
  template __global__ void k_lagrange_cell<R, 1>(KPT<R>);                    \
  template __global__ void k_lagrange_cell<R, 2>(KPT<R>);                    \
  template __global__ void k_lagrange_cell<R, 3>(KPT<R>);                    \
  MHY_LAGRANGE_INST_ONE(R, false)                                            \
  MHY_LAGRANGE_INST_ONE(R, true)
MHY_LAGRANGE_INST(double)
MHY_LAGRANGE_INST(float)
#undef MHY_LAGRANGE_INST
#undef MHY_LAGRANGE_INST_ONE

}  // namespace mhy
