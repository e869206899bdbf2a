// vl_line.hpp -- the face states and fluxes of the 1D and 2D integrators: reconstruction along a
// line of cells and the Riemann solve of one face, in the three arithmetic forms.  Included by
// translation units built with -ffp-contract=off.
#pragma once

#include <hip/hip_runtime.h>

#include "hydro_physics.hpp"
#include "vl3d_kernels.hpp"

namespace chl
{

// FindIndex, src/grid/cuda_boundaries.cu:240-302
__device__ __forceinline__ int FindIndexDev(int ig, int n, int flag, int face, int ng, double *a)
{
  if (face == 0) {
    switch (flag) {
      case 2:
        *a = -1.0;
        return 2 * ng - ig - 1;
      case 3:
        return ng;
      case 4:
        return -1;
      case 5:
        return ig;
      default:
        return ig + n - 2 * ng;
    }
  }
  switch (flag) {
    case 2:
      *a = -1.0;
      return 2 * (n - ng) - ig - 1;
    case 3:
      return n - ng - 1;
    case 4:
      return -1;
    case 5:
      return ig;
    default:
      return ig - n + 2 * ng;
  }
}

// ============================================================================ VL 1D and 2D: arithmetic forms
// The 1D and 2D integrators run in the three forms of the 3D one.  P is the form (with its
// Riemann solver): PolicyExact is the reference's order in FP64 (the oracle's bits);
// PolicyFast FP64 with the reciprocal-multiply and FMA arithmetic; PolicyMixed the
// reconstruction and Riemann fluxes in FP32, with the conserved state and its updates, the
// primitive (pressure) recovery and dt in FP64.  The mixed solvers take the split pressure
// of the 3D kernels: each face's reference p0 is the high FP32 part of its left cell's FP64
// pressure, both sides' momentum pressures are relative to it, and the normal-momentum flux
// comes back less p0, added back here in FP64 (the sum of two FP32 values, exact).

// The Riemann input of a cell's conserved values (the PCM states).  FP64 forms: the form's
// own recovery.  Mixed: the FP64 recovery, then the state in FP32; plo the low part of the
// FP64 pressure (p64 - p).
template <class P, bool DE>
__device__ __forceinline__ RState<typename P::T> SideFromCons(double d, double mx, double my, double mz, double E,
                                                              double gamma, double dge, double &plo)
{
  using T = typename P::T;
  if constexpr (sizeof(T) == sizeof(double)) {
    plo = 0.0;
    return RStateFromCons<P, DE>(d, mx, my, mz, E, gamma, dge);
  } else {
    const RState<double> s = RStateFromCons<PolicyFast, DE>(d, mx, my, mz, E, gamma, dge);
    RState<T> r{};
    r.d = T(s.d), r.mx = T(s.mx), r.my = T(s.my), r.mz = T(s.mz), r.E = T(s.E);
    r.vx = T(s.vx), r.vy = T(s.vy), r.vz = T(s.vz), r.p = T(s.p), r.inv_d = T(s.inv_d), r.dge = T(s.dge);
    plo = s.p - double(r.p);
    return r;
  }
}

// The flux of one face in FP64 from its two Riemann inputs (the split pressure's p0 added
// back to the normal-momentum flux); fge the GasEnergy flux under DE, HALF as in Hllc.
template <class P, bool DE, bool HALF = false>
__device__ __forceinline__ Cons<double> FluxFp64(const RState<typename P::T> &l, const RState<typename P::T> &r,
                                                 typename P::T gamma, double *fge)
{
  using T = typename P::T;
  T g     = T(0);
  const Cons<T> f = RiemannFlux<P, DE, HALF>(l, r, gamma, &g);
  Cons<double> o{double(f.d), double(f.mx), double(f.my), double(f.mz), double(f.E)};
  if constexpr (SplitPressure<P>) o.mx += double(l.p0);
  *fge = double(g);
  return o;
}

// The flux between two cells' PCM states a (left) and b (right), with the low parts of
// their FP64 pressures (the 3D kernels' PcmFaceFlux split).
template <class P, bool DE>
__device__ __forceinline__ Cons<double> PcmFlux(RState<typename P::T> a, double alo, RState<typename P::T> b,
                                                double blo, typename P::T gamma, double *fge)
{
  using T = typename P::T;
  if constexpr (SplitPressure<P>) {
    a.p0 = b.p0 = a.p;
    b.pd        = (b.p - a.p) + T(blo);
    a.pd        = T(alo);
  }
  return FluxFp64<P, DE, true>(a, b, gamma, fge);
}

// The interface values of the centre cell of a stencil of FP64 primitives w (in the sweep's
// frame): PLMC or PPMC in the form's precision.  pc: the centre's own pressure in that
// precision (the mixed form's face reference).
template <class P, int RK>
__device__ __forceinline__ void ReconStencil(const Prim<double> *w, double gamma, Prim<typename P::T> &L,
                                             Prim<typename P::T> &R, typename P::T &pc)
{
  using T          = typename P::T;
  constexpr int r  = ReconTraits<RK>::kRadius;
  constexpr int NS = 2 * r + 1;
  static_assert(RK == kPLMC || RK == kPPMC, "the characteristic reconstructions");
  Prim<T> s[NS];
#pragma unroll
  for (int m = 0; m < NS; m++) s[m] = {T(w[m].d), T(w[m].vx), T(w[m].vy), T(w[m].vz), T(w[m].p)};
  pc = s[r].p;
  const T g = T(gamma);
  if constexpr (RK == kPPMC && SplitPressure<P>) {
    // the mixed form's PPMC works on deviations from the centre cell (ReconPpmcCore), here
    // taken in FP64, with the centre's state for the eigenvectors; the centre is added back
    Prim<T> dv[NS];
#pragma unroll
    for (int m = 0; m < NS; m++)
      dv[m] = {T(w[m].d - w[r].d), T(w[m].vx - w[r].vx), T(w[m].vy - w[r].vy), T(w[m].vz - w[r].vz),
               T(w[m].p - w[r].p)};
    ReconPpmcCore<P>(dv, s[r], g, L, R);
    const Prim<T> &q = s[r];
    L = {L.d + q.d, L.vx + q.vx, L.vy + q.vy, L.vz + q.vz, L.p + q.p};
    R = {R.d + q.d, R.vx + q.vx, R.vy + q.vy, R.vz + q.vz, R.p + q.p};
    L.d = Fmax(L.d, T(kTinyNumber)), R.d = Fmax(R.d, T(kTinyNumber));
    L.p = Fmax(L.p, T(kTinyNumber)), R.p = Fmax(R.p, T(kTinyNumber));
  } else if constexpr (RK == kPPMC) {
    ReconPpmc<P>(s, g, L, R);
  } else {
    ReconPlmc<P>(s, g, L, R);
  }
}

// PressureFromDE with a compiled division: of the five dependent launches of a 1D dual-energy
// step the unscaled one lengthens the chain (1000 cells, PLMC, mixed: 28.0 against 28.6 us).
__device__ __forceinline__ double LinePressureFromDE(double E, double U_total, double U_advected, double gamma)
{
  const double U = (U_total / E > kDeEta1) ? U_total : U_advected;
  return Fmax(U * (gamma - 1.0), kTinyNumber);
}

// The interface values of cell c from the conserved half state W (fields nf apart) along a
// line of stride st, whose normal and transverse momenta are the fields o1, o2, o3:
// primitives as Load_Data forms them (PLMC, PPMC) or as PLMP_cuda does
// (plmp_cuda.cu:104-120), in FP64, then the reconstruction in the form's precision; PCM
// passes the conserved values through in the exact form (pcm_cuda.cu:13-97) and the
// primitives in the others.  With dual energy (PLMC and PPMC only) the pressure is
// Load_Data's DE pressure and the specific GasEnergy is reconstructed beside
// (reconstruction.h:179-191, plmc_cuda.cu, ppmc_cuda.cu:668-672).  pc: the cell's own
// pressure in the form's precision (the mixed form's face reference).
template <class P, int RK, bool DE = false>
__device__ __forceinline__ void ReconLine(const double *W, long nf, long c, long st, int o1, int o2, int o3,
                                          double gamma, Prim<typename P::T> &L, Prim<typename P::T> &R,
                                          typename P::T &geL, typename P::T &geR, typename P::T &pc)
{
  using T          = typename P::T;
  constexpr int r  = ReconTraits<RK>::kRadius;
  constexpr int NS = 2 * r + 1;
  static_assert(!DE || RK != kPCM, "the PCM states carry the conserved GasEnergy (Vl2dPcmFluxKernel)");
  Prim<T> s[NS];
  Prim<double> w[NS];  // the FP64 primitives (the forms other than the exact PCM pass-through)
  T ge[NS];
#pragma unroll
  for (int m = 0; m < NS; m++) {
    const long q   = c + long(m - r) * st;
    const double d = W[q], mx = W[o1 * nf + q], my = W[o2 * nf + q], mz = W[o3 * nf + q], E = W[4 * nf + q];
    if constexpr (RK == kPCM && P::kExact) {
      s[m] = {d, mx, my, mz, E};
      continue;
    } else if constexpr (RK == kPLMP || RK == kPPMP) {
      const double vx = mx / d, vy = my / d, vz = mz / d;
      if constexpr (DE) {  // plmp_cuda.cu:116-121
        const double g = W[5 * nf + q], E_kin = 0.5 * d * (vx * vx + vy * vy + vz * vz);
        w[m]  = {d, vx, vy, vz, LinePressureFromDE(E, E - E_kin, g, gamma)};
        ge[m] = T(g / d);
      } else {
        w[m] = {d, vx, vy, vz, Fmax((E - 0.5 * d * (vx * vx + vy * vy + vz * vz)) * (gamma - 1.0), kTinyNumber)};
      }
    } else if constexpr (DE) {
      const double vx = mx / d, vy = my / d, vz = mz / d, g = W[5 * nf + q];
      w[m]  = {d, vx, vy, vz, LinePressureFromDE(E, E - 0.5 * d * SquareMag(vx, vy, vz), g, gamma)};
      ge[m] = T(g / d);
    } else {
      w[m] = LoadPrim(d, mx, my, mz, E, gamma);
    }
    s[m] = {T(w[m].d), T(w[m].vx), T(w[m].vy), T(w[m].vz), T(w[m].p)};
  }
  if constexpr (RK == kPPMC || RK == kPLMC) {
    ReconStencil<P, RK>(w, gamma, L, R, pc);
    if constexpr (DE && RK == kPPMC) ReconPpmcScalar<P>(ge, geL, geR);
    if constexpr (DE && RK == kPLMC) ReconPlmcScalar<P>(ge, geL, geR);
    return;
  }
  pc = s[r].p;
  if constexpr (RK == kPCM) {
    L = R = s[0];
  } else if constexpr (RK == kPLMP) {
    ReconPlmp<P>(s, L, R);
    if constexpr (DE) ReconPlmpScalar<P>(ge, geL, geR);
  } else if constexpr (RK == kPPMP) {
    ReconPpmp<P>(s, L, R);
    if constexpr (DE) ReconPpmpScalar<P>(ge, geL, geR);
  }
}

// The flux of the face between a cell whose interface value there is L and the next cell,
// whose value there is R; p0 the left cell's own pressure (the mixed form's reference).
template <class P, int RK, bool DE>
__device__ __forceinline__ Cons<double> ReconFlux(const Prim<typename P::T> &L, const Prim<typename P::T> &R,
                                                  typename P::T geL, typename P::T geR, typename P::T p0,
                                                  typename P::T gamma, typename P::T inv_gm1, double *fge)
{
  using T = typename P::T;
  RState<T> l, r;
  if constexpr (SplitPressure<P>) {
    Prim<T> a = L, b = R;
    a.p       = Fmax(L.p, T(kTinyNumber));
    b.p       = Fmax(R.p, T(kTinyNumber));
    l         = RStateFromPrim<P, DE>(a, gamma, inv_gm1, geL);
    r         = RStateFromPrim<P, DE>(b, gamma, inv_gm1, geR);
    l.p0 = r.p0 = p0;
    l.pd        = Fmax(l.p - p0, -p0);
    r.pd        = Fmax(r.p - p0, -p0);
  } else {
    l = IfaceState<P, RK, DE>(L, gamma, inv_gm1, geL);
    r = IfaceState<P, RK, DE>(R, gamma, inv_gm1, geR);
  }
  return FluxFp64<P, DE>(l, r, gamma, fge);
}

}  // namespace chl
