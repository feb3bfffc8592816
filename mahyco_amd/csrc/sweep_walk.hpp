// Remap sweeps along y with one lane per column (Remap::computeGradPhiFace,
// computeGradPhi, computeUpwindFaceQuantitiesForProjection, computeUremap of
// the y direction; remap/PhaseRemap1.cc, remap/PhaseRemap2.cc).
//
// A wave covers 64 consecutive columns and walks down a band of
// kp.walkRows rows, plus two halo rows above and below.  Every row access of the wave
// is a whole 64-cell row segment.  Each iteration loads one new row and
// keeps the two before it in registers: the divided difference at the new
// row's minus face, the slope (or the PenteBorne fluxes) of the row before,
// the face value between the two rows before, and the update of the row
// two back.  Operation order is that of the wave-strip sweeps (and of the
// reference), so FP64 results are bitwise the same.
//
// LAG: the first sweep of a step with the cell part of the Lagrange phase, as the
// strips have it: a row's remap vector waits two iterations in a ring of three slots per
// thread in LDS, and only the band's own rows store what outlives the step.
#pragma once

#include <type_traits>

#include "final_math.hpp"
#include "kernels.hpp"
#include "lagrange_cell.hpp"
#include "sweep_math.hpp"
#include "sweep_update.hpp"

namespace mhy {

using namespace sw;

namespace {

// end-of-Lagrange node position (updatePosition, PhaseLagrange.cc:203-208)
template <class R>
__device__ __forceinline__ D2 lagNodeK(const KPT<R>& kp, double dt1, long j, long i) {
  const long p = j * (kp.o.nx + 1) + i;
  const D2 e = eulerNode(kp.o, j, i);
  return {e.x + (double)at(kp.ul, p) * dt1, e.y + (double)at(kp.vl, p) * dt1};
}

// width across the y-sweep faces (HvLagrange, PhaseRemap2.cc): right then
// left face
template <class R>
__device__ __forceinline__ double widthY(const KPT<R>& kp, double dt1, long j, long i) {
  double h = 0.;
  h += 0.5 * d2norm(d2sub(lagNodeK(kp, dt1, j + 1, i + 1), lagNodeK(kp, dt1, j, i + 1)));
  h += 0.5 * d2norm(d2sub(lagNodeK(kp, dt1, j + 1, i), lagNodeK(kp, dt1, j, i)));
  return h;
}

}  // namespace

// b: linear block index; the waves of all bands are numbered column-group
// first, 4 per block.
template <class R, int M, bool PP, class P, bool LAG = false>
__device__ __forceinline__ void sweepWalkYBody(const KPT<R>& kp, unsigned b) {
  using T = typename std::conditional<kMixed<R> && !PP, float, double>::type;
  constexpr int NC = 3 * M + 1;
  constexpr bool kF32 = sizeof(T) == 4;
  const Opts& o = kp.o;
  const auto& f = kp.f;
  const long nx = o.nx, ny = o.ny;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long ngx = (nx + 63) / 64;
  const long g = (long)b * 4 + wave;
  const long i0 = (g % ngx) * 64 + lane;
  const int rows = kp.walkRows;
  const long a0 = (g / ngx) * rows;

  double* const* Uin = (P::sweep(kp) == 1) ? f.UL : f.U1;
  const double dtn = f.sc->dt[kp.cur], dt1 = f.sc->dt[kp.nxt];
  const bool needH = PP || P::limiter(o) >= MHY_LIM_MINMODG;
  const bool mixteOpt = PP && P::mixte(o);
  const bool pb = PP && P::methode(o) == 2;
  const bool formed = P::order(o) > 1;
  const R* uy = kp.vl;

  // rolling state: A = row r-2, B = row r-1
  T phA[NC], phB[NC], dMB[NC], gA[NC], avA[NC], faceA[NC], dualA[M];
#pragma unroll
  for (int q = 0; q < NC; ++q) phA[q] = phB[q] = dMB[q] = gA[q] = avA[q] = faceA[q] = T(0.0);
#pragma unroll
  for (int k = 0; k < M; ++k) dualA[k] = T(0.0);
  double xcA = 0.0, xcB = 0.0, vA = 0.0, vB = 0.0;
  T HA = T(0.0), HB = T(0.0);
  int flA = 0, flB = 0;

  // LAG: the remap vectors of the last three rows, each thread its own slots
  __shared__ double uRing[LAG ? 3 : 1][LAG ? NC : 1][LAG ? 256 : 1];
  int slot = 0;  // ring slot of the new row

  for (int k = 0; k < rows + 4; ++k) {
    // the column and what derives from it (addresses, Euler coordinates) are
    // formed again for every row from an opaque copy of the index: hoisted
    // out of the loop they would hold registers through every row
    int iop = (int)i0;
    asm volatile("" : "+v"(iop));
    const long i = iop;
    const bool inT = (i < nx);
    // row r of this lane's column: Phi, centroid, width, flags
    auto loadRow = [&](long r, T* ph, double& x, T& h, int& flg) {
      const long cb = r * nx + i;
      double u[NC];
      if constexpr (LAG) {
        // the Lagrange update of the cell; a band's own rows store what outlives the step
        const bool own = r >= a0 && r < a0 + rows;
        LagCell<M> lc;
        lagrangeCellCompute<R, M, P>(kp, cb, r, i, own, lc);
#pragma unroll
        for (int q = 0; q < NC; ++q) u[q] = lc.U[q], uRing[slot][q][threadIdx.x] = lc.U[q];
        cellPhi<M, PP, T>(u, lc.V, lc.q, ph);
        x = lc.xc.y;
        if (own) at(f.VL, cb) = lc.V, at(f.XcL, cb) = lc.xc.x;
        h = needH ? T(widthY(kp, dt1, r, i)) : T(0.0);
        flg = 0;
        return;
      }
      const int nload = PP ? 3 * M : NC;
#pragma unroll
      for (int q = 0; q < NC; ++q) u[q] = (q < nload) ? at(Uin[q], cb) : 0.0;
      cellPhi<M, PP, T>(u, PP ? 1.0 : at(f.VL, cb), PP ? at(f.qL, cb) : 0.0, ph);
      x = at(f.YcL, cb);
      h = needH ? T(widthY(kp, dt1, r, i)) : T(0.0);
      flg = 0;
      if (mixteOpt) flg = (P::sweep(kp) == 1) ? packFlags(cellMixed(at(f.flags, cb)), cellPure(at(f.flags, cb))) : packedFlags<M, T>(ph);
    };
    // normal velocity of face r, between rows r-1 and r (PrepareRemap.cc:50-62)
    auto fnv = [&](long r) {
      const long n1 = r * (nx + 1) + i, n2 = n1 + 1;
      return 0.0 + ((0.0 + (double)at(uy, n1)) + (double)at(uy, n2)) * 0.5;
    };
    const long r = a0 - 2 + k, rB = r - 1, rA = r - 2;
    // new row N
    T phN[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) phN[q] = T(0.0);
    double xcN = 0.0;
    T HN = T(0.0);
    int flN = 0;
    if (inT && r >= 0 && r < ny) loadRow(r, phN, xcN, HN, flN);
    const double vN = (inT && r >= 0 && r <= ny) ? fnv(r) : 0.0;

    // divided difference at the minus face of row N (between rows B and N)
    T dMN[NC];
    {
      const bool inMN = (r >= 1);
      const T xcmT = kF32 ? T(xcB - xcN) : T(xcB), xcT = kF32 ? T(0.0) : T(xcN);
      const Nbr<T> nN{phB, phN, phN, xcmT, xcT, xcT, inMN, false, HN, HB, HN, false};
#pragma unroll
      for (int q = 0; q < NC; ++q) dMN[q] = formed ? faceDiffM<false, T>(nN, q) : T(0.0);
    }

    // row B with its neighbours A and N; a missing neighbour takes row B's
    // values (PhaseRemap1.cc:157-158)
    const bool inB = inT && rB >= 0 && rB < ny;
    const bool inMB = (rB >= 1), inPB = (rB + 1 < ny);
    T phmB[NC], phpB[NC], dPB[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      phmB[q] = inMB ? phA[q] : phB[q];
      phpB[q] = inPB ? phN[q] : phB[q];
      dPB[q] = inPB ? dMN[q] : T(0.0);
    }
    const double xcmB = inMB ? xcA : xcB, xcpB = inPB ? xcN : xcB;
    const T HmB = inMB ? HA : HB, HpB = inPB ? HN : HB;
    const int fmB = inMB ? flA : flB, fpB = inPB ? flN : flB;
    const T xcmT = kF32 ? T(xcmB - xcB) : T(xcmB), xcT = kF32 ? T(0.0) : T(xcB);
    const T xcpT = kF32 ? T(xcpB - xcB) : T(xcpB);
    Nbr<T> nB{phmB, phB, phpB, xcmT, xcT, xcpT, inMB, inPB, HB, HmB, HpB, false};
    if (mixteOpt) nB.vp = ((flB >> 8) == 0) && flB == fpB && flB == fmB;
    nB.dM = dMB;
    nB.dP = dPB;

    // face value at the minus face of row B (between rows A and B)
    T faceB[NC], gB[NC], avB[NC], dualB[M];
#pragma unroll
    for (int q = 0; q < NC; ++q) faceB[q] = gB[q] = avB[q] = T(0.0);
#pragma unroll
    for (int k2 = 0; k2 < M; ++k2) dualB[k2] = T(0.0);
    if (!PP) {
#pragma unroll
      for (int q = 0; q < NC; ++q) gB[q] = inB ? gradQ<false, PP, P, T>(o, nB, q) : T(0.0);
      // upwind value (UtilesRemap-Impl.h:491-501); y: back = above (row B),
      // front = below (row A)
      const double dxl = xcA - xcB;  // front - back
      const bool upLo = !(vB * dxl > 0.0);
      const double xf = 0.5 * (o.dy * (double)rB + o.dy * (double)rB);
      const T s = T(0.0 + (xf - (upLo ? xcA : xcB)));
#pragma unroll
      for (int q = 0; q < NC; ++q) faceB[q] = upLo ? phA[q] + gA[q] * s : phB[q] + gB[q] * s;
    } else {
      T arB[NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) arB[q] = T(0.0);
      if (formed && inB) ppFluxes<M, false, P, T>(o, nB, T(vB), T(vN), T(dtn), pb, arB, avB, dualB);
#pragma unroll
      for (int q = 0; q < NC; ++q) faceB[q] = formed ? avA[q] - arB[q] : T(0.0);
    }

    // update of row A: minus face faceA, plus face faceB
    if (inT && rA >= a0 && rA < a0 + rows && rA < ny) {
      const long c = rA * nx + i;
      const bool hasM = (rA >= 1), hasP = (rA + 1 < ny);
      // Euler length of a face (Init.cc:528-533): the norm of an edge along one
      // axis, sqrt(fl(w w)) = |w| in binary floating point
      const double Lm = fabs(o.dx * (double)(i + 1) - o.dx * (double)i), Lp = Lm;
      T phiM[NC], phiP[NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        phiM[q] = hasM ? faceA[q] : T(0.0);
        phiP[q] = hasP ? faceB[q] : T(0.0);
      }
      if (pb) {
        const double w = (Lm + Lp) * 0.5;
#pragma unroll
        for (int k2 = 0; k2 < M; ++k2) at(f.DF[k2], c) = formed ? (double)dualA[k2] * w : 0.0;
      }
      double uOwn[LAG ? NC : 1];
      if constexpr (LAG) {
        const int sA = slot == 2 ? 0 : slot + 1;  // two rows ago
#pragma unroll
        for (int q = 0; q < NC; ++q) uOwn[q] = uRing[sA][q][threadIdx.x];
      }
      sweepUpdateCell<R, M, PP, false, P, T>(kp, c, i, rA, rA, hasM, hasP, vA, vB, Lm, Lp, phiM, phiP, LAG ? uOwn : nullptr);
    }

    // rotate: B becomes A, N becomes B
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      phA[q] = phB[q], phB[q] = phN[q];
      dMB[q] = dMN[q];
      gA[q] = gB[q];
      avA[q] = avB[q];
      faceA[q] = faceB[q];
    }
#pragma unroll
    for (int k2 = 0; k2 < M; ++k2) dualA[k2] = dualB[k2];
    xcA = xcB, xcB = xcN;
    HA = HB, HB = HN;
    flA = flB, flB = flN;
    vA = vB, vB = vN;
    if constexpr (LAG) slot = slot == 2 ? 0 : slot + 1;
  }
}

// waves per SIMD the walker is compiled for: 4 for one material with limited
// slopes (128 VGPRs, a few spilled; unbounded it takes 136 and runs 3 waves)
template <class R, int M, bool PP>
constexpr int kWalkWaves = (M == 1 && !PP) ? 4 : 1;

template <class R, int M, bool PP, class P>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kWalkWaves<R, M, PP>))) void k_sweep_walk(
    KPT<R> kp) {
  sweepWalkYBody<R, M, PP, P>(kp, blockIdx.x);
}

// the first sweep of a step with the cell part of the Lagrange phase.  FP64: 166 VGPRs
// (3 waves per SIMD), 207, 253 for 1, 2, 3 materials; mixed 138, 165, 191.  Held to 4
// waves it spills: 4096^2 1630 -> 2105 us a step, 2048^2 mixed 402 -> 409.
template <class R, int M, class P>
__global__ __launch_bounds__(256) void k_sweep_walk_lag(KPT<R> kp) {
  sweepWalkYBody<R, M, false, P, true>(kp, blockIdx.x);
}

template <class R, int M, bool PP, bool ONE>
__global__ __launch_bounds__(256) void k_sweep_walk_batch(BatchLaunchT<R> bl) {
  batchRun<ONE>(bl, [&](const KPT<R>& kp, unsigned local, unsigned, unsigned) {
    sweepWalkYBody<R, M, PP, RunOpts>(kp, local);
  });
}

}  // namespace mhy
