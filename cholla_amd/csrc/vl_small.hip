// vl_small.hip -- the 1D and 2D van Leer steps of hydro boxes with HLLC and PLMC or PPMC (no dual
// energy, no gravity), fused: a batch of 1D steps is one launch and a 2D step two.  The other
// options run the unfused kernels of support_kernels.hip; every face state, flux and update
// here is formed by the same functions in the same order, so the results are the same bits.
//
// Built with -ffp-contract=off, as support_kernels.hip is.
#include <hip/hip_runtime.h>

#include "support_kernels.hpp"
#include "vl_line.hpp"

namespace chl
{

// ============================================================================ 1D: a batch of steps in one launch
// A 1D box of at most 1024 cells fits one workgroup, and a step of it is a chain of five short
// phases (dt; PCM fluxes; half state; reconstruction; fluxes; update and ghosts): four launches
// of 1.4-9.7 us with gaps between them, most of each spent starting up.  Here one workgroup
// keeps the state in LDS and runs every step of a batch, a barrier between phases, one cell
// (CELLS: up to two) per thread.  Each face is solved and each cell reconstructed once; the
// unfused stage 2 reconstructs three cells per thread.  What bounds it is the latency of the
// dependent FP64 chain of a reconstruction and a solve on one or two waves per SIMD.  Sod, 100
// cells, PLMC, reference order: 26.6 -> 4.5 us a step.  The limit of 1024 cells is the LDS's (15
// doubles a cell, 120 of its 160 KB) and two cells a thread, not a crossover: 1024 cells (ghosts
// included) take 12.3 us a step here, 1025 in the unfused launches 23.6, and 4008 there 24.2.
constexpr int kLineThreads = 512;

template <class P, int RK, int CELLS>
__global__ void __launch_bounds__(kLineThreads) Vl1dRunKernel(double *U, int n, int ng, double dx, double gamma,
                                                              GhostFlags fl, int n_steps, int first, double t0,
                                                              double tout, double cfl, LineClock *clk)
{
  using T            = typename P::T;
  constexpr int NMAX = kLineThreads * CELLS;
  constexpr int r    = ReconTraits<RK>::kRadius;
  __shared__ double a[5][NMAX];  // the conserved state
  __shared__ double b[5][NMAX];  // half-step primitives, then the fluxes of the full update
  __shared__ double c[5][NMAX];  // stage-1 fluxes, then each cell's lower interface value
  __shared__ double red[kLineThreads / 64];
  const int tid = threadIdx.x, nt = blockDim.x;
  const T g = T(gamma), inv_gm1 = P::kExact ? T(RcpRefined(gamma - 1.0)) : T(1.0 / (gamma - 1.0));
  for (int id = tid; id < n; id += nt)
    for (int f = 0; f < 5; f++) a[f][id] = U[size_t(f) * n + id];
  __syncthreads();
  auto real = [&](int id) { return id >= ng && id < n - ng; };
  // the inverse crossing time of a cell (Calc_dt_1D, hydro_cuda.cu:437-472)
  auto crossing = [&](int id) {
    const double d = a[0][id], dinv = 1.0 / d;
    const double vx = a[1][id] * dinv, vy = a[2][id] * dinv, vz = a[3][id] * dinv;
    const double pr = Fmax((a[4][id] - 0.5 * d * (vx * vx + vy * vy + vz * vz)) * (gamma - 1.0), kTinyNumber);
    return (Fabs(vx) + __builtin_sqrt(dinv * gamma * pr)) / dx;
  };
  // the workgroup's maximum, to every thread; ends with every earlier LDS write visible
  auto block_max = [&](double m) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = Fmax(m, __shfl_xor(m, off, 64));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    double v = red[0];
    for (int w = 1; w < nt >> 6; w++) v = Fmax(v, red[w]);
    return v;
  };
  auto side = [&](int id, double &plo) {
    return SideFromCons<P, false>(a[0][id], a[1][id], a[2][id], a[3][id], a[4][id], gamma, 0.0, plo);
  };
  double t = t0, dt = 0.0, dti;
  int taken = 0;
  if (first) {
    double m = 0.0;
    for (int id = tid; id < n; id += nt)
      if (real(id)) m = Fmax(m, crossing(id));
    dti = block_max(m);
  } else {
    dti = __longlong_as_double((long long)clk->dti), t = clk->t, taken = clk->nstep;
  }
  for (int s = 0; s < n_steps; s++) {
    // DtAdvanceKernel's arithmetic (main.cpp:254-261)
    dt = cfl / dti;
    if (t + dt > tout) dt = tout - t;
    if (!(t < tout)) dt = 0.0;
    t += dt;
    if (dt > 0.0) taken++;
    if (dt == 0.0) break;  // past the output time: the state stays as it is
    const double half = 0.5 * dt / dx, full = dt / dx;
    double unused;
    for (int id = tid; id < n - 1; id += nt) {  // PCM fluxes of the faces id + 1/2
      double plo, qlo;
      const RState<T> l = side(id, plo), q = side(id + 1, qlo);
      const Cons<double> f = PcmFlux<P, false>(l, plo, q, qlo, g, &unused);
      c[0][id] = f.d, c[1][id] = f.mx, c[2][id] = f.my, c[3][id] = f.mz, c[4][id] = f.E;
    }
    __syncthreads();
    for (int id = tid; id < n; id += nt)
      if (id >= 1 && id < n - 1) {
        double u[5];
#pragma unroll
        for (int f = 0; f < 5; f++) u[f] = a[f][id] + half * (c[f][id - 1] - c[f][id]);
        const Prim<double> w = LoadPrim(u[0], u[1], u[2], u[3], u[4], gamma);
        b[0][id] = w.d, b[1][id] = w.vx, b[2][id] = w.vy, b[3][id] = w.vz, b[4][id] = w.p;
      }
    __syncthreads();
    Prim<T> L[CELLS];
    T pc[CELLS];
#pragma unroll
    for (int q = 0; q < CELLS; q++) {
      const int id = tid + q * nt;
      if (id >= ng - 1 && id <= n - ng) {
        Prim<double> w[2 * r + 1];
#pragma unroll
        for (int m = 0; m < 2 * r + 1; m++) {
          const int k = id - r + m;
          w[m]        = {b[0][k], b[1][k], b[2][k], b[3][k], b[4][k]};
        }
        Prim<T> R;
        ReconStencil<P, RK>(w, gamma, L[q], R, pc[q]);
        c[0][id] = double(R.d), c[1][id] = double(R.vx), c[2][id] = double(R.vy), c[3][id] = double(R.vz);
        c[4][id] = double(R.p);
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < CELLS; q++) {
      const int id = tid + q * nt;
      if (id >= ng - 1 && id < n - ng) {  // the face id + 1/2
        const Prim<T> R{T(c[0][id + 1]), T(c[1][id + 1]), T(c[2][id + 1]), T(c[3][id + 1]), T(c[4][id + 1])};
        const Cons<double> f = ReconFlux<P, RK, false>(L[q], R, T(0), T(0), pc[q], g, inv_gm1, &unused);
        b[0][id] = f.d, b[1][id] = f.mx, b[2][id] = f.my, b[3][id] = f.mz, b[4][id] = f.E;
      }
    }
    __syncthreads();
    double m = 0.0;
    for (int id = tid; id < n; id += nt)
      if (real(id)) {
#pragma unroll
        for (int f = 0; f < 5; f++) a[f][id] = a[f][id] + full * (b[f][id - 1] - b[f][id]);
        m = Fmax(m, crossing(id));
      }
    dti = block_max(m);
    for (int id = tid; id < n; id += nt)  // the two ghost slabs (GhostFillKernel)
      if (!real(id)) {
        double sgn  = 1.0;
        const int lo = id < ng, src = FindIndexDev(id, n, fl.f[lo ? 0 : 1], lo ? 0 : 1, ng, &sgn);
        double u[5];
#pragma unroll
        for (int f = 0; f < 5; f++) u[f] = a[f][src];
        if (fl.f[0] == 2 || fl.f[1] == 2) u[1] *= sgn;
        if (fl.f[lo ? 0 : 1] == 3 && (lo ? u[1] > 0.0 : u[1] < 0.0)) {
          u[4] -= 0.5 * (u[1] * u[1]) / u[0];
          u[1] = 0.0;
        }
#pragma unroll
        for (int f = 0; f < 5; f++) a[f][id] = u[f];
      }
    __syncthreads();
  }
  for (int id = tid; id < n; id += nt)
    for (int f = 0; f < 5; f++) U[size_t(f) * n + id] = a[f][id];
  if (tid == 0) {
    clk->dti = (unsigned long long)__double_as_longlong(dti), clk->dt = dt, clk->t = t;
    clk->nstep = taken;
  }
}

template <class P, int RK>
static hipError_t LaunchVl1dRunP(double *U, int n, int ng, double dx, double gamma, const int flags[6], int n_steps,
                                 bool first, double t0, double tout, double cfl, LineClock *clk, hipStream_t s)
{
  GhostFlags fl;
  for (int q = 0; q < 6; q++) fl.f[q] = flags[q];
  fl.diode = 1;
  const int cells = n <= kLineThreads ? 1 : 2;
  const dim3 block(unsigned(((n + cells - 1) / cells + 63) / 64 * 64));
  if (cells == 1) {
    hipLaunchKernelGGL((Vl1dRunKernel<P, RK, 1>), dim3(1), block, 0, s, U, n, ng, dx, gamma, fl, n_steps, int(first), t0,
                       tout, cfl, clk);
  } else {
    hipLaunchKernelGGL((Vl1dRunKernel<P, RK, 2>), dim3(1), block, 0, s, U, n, ng, dx, gamma, fl, n_steps, int(first), t0,
                       tout, cfl, clk);
  }
  return hipGetLastError();
}

bool Vl1dRunTakes(int n, int recon, int riemann, bool de, const GravSpec &grav)
{
  return n <= 2 * kLineThreads && (recon == kPLMC || recon == kPPMC) && riemann == kRiemannHllc && !de && grav.id == 0;
}

// A form's launch of fn<P, RK>: PLMC or PPMC.
#define CHL_SMALL_FORM(fn, ...)                                                                       \
  switch (form) {                                                                                     \
    case PolicyExact::kId:                                                                            \
      return recon == kPPMC ? fn<PolicyExact, kPPMC>(__VA_ARGS__) : fn<PolicyExact, kPLMC>(__VA_ARGS__); \
    case PolicyFast::kId:                                                                             \
      return recon == kPPMC ? fn<PolicyFast, kPPMC>(__VA_ARGS__) : fn<PolicyFast, kPLMC>(__VA_ARGS__);   \
    case PolicyMixed::kId:                                                                            \
      return recon == kPPMC ? fn<PolicyMixed, kPPMC>(__VA_ARGS__) : fn<PolicyMixed, kPLMC>(__VA_ARGS__); \
  }                                                                                                   \
  return hipErrorInvalidValue

hipError_t LaunchVl1dRun(double *U, int n, int ng, int recon, int form, double dx, double gamma, const int flags[6],
                         int n_steps, bool first, double t0, double tout, double cfl, LineClock *clk, hipStream_t s)
{
  if (n > 2 * kLineThreads || n < 2 * ng + 1 || (recon != kPLMC && recon != kPPMC)) return hipErrorInvalidValue;
  CHL_SMALL_FORM(LaunchVl1dRunP, U, n, ng, dx, gamma, flags, n_steps, first, t0, tout, cfl, clk, s);
}

// ============================================================================ 2D: two launches a step
// A 2D box is a few hundred workgroups, so its step is bound by the latency of each launch's
// chain, and by what the unfused launches repeat: every face reconstructed its two cells from
// ten conserved cells, and fluxes went through memory.  Stage 1 and stage 2 here are tiles:
// half of a workgroup's threads take the x sweep of the tile's cells and half the y sweep, so a
// thread's chain is one reconstruction and one solve; neighbours exchange through LDS, and the
// tile's last row and column (and in stage 2 its first) only feed the others.  Periodic boxes
// write their ghost images from the update.  KH 320x192, PPMC, fast form: stage 2 13.5 us
// and stage 1 7.6, against 16.8 + 6.5 and 5.5 + 5.8 for the pairs of launches they replaced, and
// no ghost fill (4.4); a step 33 us against 51.

// Stage 1: PCM states and HLLC on the lower x and y faces of a 32 x 8 tile of cells, the dt/2
// update of its 31 x 7 cells whose upper faces it holds too (Update_Conserved_Variables_2D_half,
// VL_2D_cuda.cu:183-256), stored as density, velocities and energy (the sweeps' pressures differ
// in their last bit by direction).  Cells [1, n - 2] on both axes.
constexpr int kS1X = 32, kS1Y = 8, kS1Cells = kS1X * kS1Y;

template <class P>
__global__ void __launch_bounds__(2 * kS1Cells) Vl2dStage1Kernel(const double *U, double *W, int nx, int ny, double dx,
                                                                 double dy, const double *dt_dev, double dt_host,
                                                                 double gamma, unsigned long long *dti_reset)
{
  using T       = typename P::T;
  const long nc = long(nx) * ny;
  __shared__ double f[2][5][kS1Y][kS1X];
  if (dti_reset && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *dti_reset = 0ull;
  const int dir = threadIdx.x / kS1Cells, c = threadIdx.x % kS1Cells;
  const int tx = c % kS1X, ty = c / kS1X;
  const int i = 1 + int(blockIdx.x) * (kS1X - 1) + tx, j = 1 + int(blockIdx.y) * (kS1Y - 1) + ty;
  const bool in = i < nx && j < ny;
  const long id = in ? i + long(j) * nx : 0;
  double u[5] = {};
  if (in) {
    const long lo = id - (dir ? nx : 1);
    const int o1 = dir ? 2 : 1, o2 = dir ? 3 : 2, o3 = dir ? 1 : 3;
#pragma unroll
    for (int q = 0; q < 5; q++) u[q] = U[q * nc + id];
    double alo, blo, unused;
    const RState<T> l = SideFromCons<P, false>(U[lo], U[o1 * nc + lo], U[o2 * nc + lo], U[o3 * nc + lo], U[4 * nc + lo],
                                               gamma, 0.0, alo);
    const RState<T> r = SideFromCons<P, false>(u[0], dir ? u[2] : u[1], dir ? u[3] : u[2], dir ? u[1] : u[3], u[4],
                                               gamma, 0.0, blo);
    const Cons<double> v = PcmFlux<P, false>(l, alo, r, blo, T(gamma), &unused);
    f[dir][0][ty][tx] = v.d, f[dir][o1][ty][tx] = v.mx, f[dir][o2][ty][tx] = v.my, f[dir][o3][ty][tx] = v.mz;
    f[dir][4][ty][tx] = v.E;
  }
  __syncthreads();
  if (dir || !in || tx == kS1X - 1 || ty == kS1Y - 1 || i >= nx - 1 || j >= ny - 1) return;
  const double dt = 0.5 * (dt_dev ? *dt_dev : dt_host), dtodx = dt / dx, dtody = dt / dy;
#pragma unroll
  for (int q = 0; q < 5; q++)
    u[q] = u[q] + dtodx * (f[0][q][ty][tx] - f[0][q][ty][tx + 1]) + dtody * (f[1][q][ty][tx] - f[1][q][ty + 1][tx]);
  const double rd = RcpRefined(u[0]);
  W[id] = u[0], W[nc + id] = Quot(u[1], u[0], rd), W[2 * nc + id] = Quot(u[2], u[0], rd);
  W[3 * nc + id] = Quot(u[3], u[0], rd), W[4 * nc + id] = u[4];
}

// Stage 2: reconstruction of a 32 x 12 tile of cells along x and y, HLLC on their upper faces,
// and the full update of the 30 x 10 cells inside (Update_Conserved_Variables_2D,
// hydro_cuda.cu:84-160) with the next inverse dt (Calc_dt_2D, :474-510) and, for periodic boxes,
// the ghost images.  The half state of the tile and its stencil is staged in LDS with the
// pressures of both sweeps.
constexpr int kS2X = 32, kS2Y = 12, kS2Cells = kS2X * kS2Y;

template <class P, int RK>
__global__ void __launch_bounds__(2 * kS2Cells) Vl2dStage2Kernel(double *U, const double *W, int nx, int ny, int ng,
                                                                 double dx, double dy, const double *dt_dev,
                                                                 double dt_host, double gamma, int periodic,
                                                                 unsigned long long *dti)
{
  using T          = typename P::T;
  constexpr int r  = ReconTraits<RK>::kRadius, NT = 2 * kS2Cells;
  constexpr int SX = kS2X + 2 * r, SY = kS2Y + 2 * r;
  const long nc    = long(nx) * ny;
  __shared__ double w[6][SY * SX];        // d, vx, vy, vz, pressure of the x sweep, of the y sweep
  __shared__ T lower[2][5][kS2Cells];     // each cell's interface values at its lower x / y face
  __shared__ double f[2][5][kS2Y][kS2X];  // fluxes of its upper x / y face
  __shared__ double red[NT / 64];
  const int tid = threadIdx.x, dir = tid / kS2Cells, c = tid % kS2Cells, tx = c % kS2X, ty = c / kS2X;
  // the tile's first cell: one before its first updated one
  const int i0 = ng - 1 + int(blockIdx.x) * (kS2X - 2), j0 = ng - 1 + int(blockIdx.y) * (kS2Y - 2);
  for (int q = tid; q < SX * SY; q += NT) {
    const int i = i0 - r + q % SX, j = j0 - r + q / SX;
    if (i < 1 || j < 1 || i > nx - 2 || j > ny - 2) continue;  // no half state, and no stencil reads it
    const long id = i + long(j) * nx;
    const double d = W[id], vx = W[nc + id], vy = W[2 * nc + id], vz = W[3 * nc + id], E = W[4 * nc + id];
    w[0][q] = d, w[1][q] = vx, w[2][q] = vy, w[3][q] = vz;
    w[4][q] = PressureFromCons(E, d, vx, vy, vz, gamma);  // Load_Data in each sweep's frame
    w[5][q] = PressureFromCons(E, d, vy, vz, vx, gamma);
  }
  __syncthreads();
  const int i = i0 + tx, j = j0 + ty;
  // along the sweep and across it: cells whose interfaces some updated cell of the box needs
  const int along = dir ? j : i, across = dir ? i : j, na = dir ? ny : nx, nb = dir ? nx : ny;
  const bool take = along <= na - ng && across >= ng && across < nb - ng;
  const int o1 = dir ? 2 : 1, o2 = dir ? 3 : 2, o3 = dir ? 1 : 3;
  const T g = T(gamma), inv_gm1 = P::kExact ? T(RcpRefined(gamma - 1.0)) : T(1.0 / (gamma - 1.0));
  Prim<T> L;
  T pc = T(0);
  if (take) {
    const int st = dir ? SX : 1, first = (ty + r) * SX + tx + r - r * st;
    Prim<double> s[2 * r + 1];
#pragma unroll
    for (int m = 0; m < 2 * r + 1; m++) {
      const int q = first + m * st;
      s[m]        = {w[0][q], w[o1][q], w[o2][q], w[o3][q], w[4 + dir][q]};
    }
    Prim<T> R;
    ReconStencil<P, RK>(s, gamma, L, R, pc);
    lower[dir][0][c] = R.d, lower[dir][1][c] = R.vx, lower[dir][2][c] = R.vy;
    lower[dir][3][c] = R.vz, lower[dir][4][c] = R.p;
  }
  __syncthreads();
  if (take && along < na - ng && (dir ? ty < kS2Y - 1 : tx < kS2X - 1)) {
    const int n = c + (dir ? kS2X : 1);
    const Prim<T> R{lower[dir][0][n], lower[dir][1][n], lower[dir][2][n], lower[dir][3][n], lower[dir][4][n]};
    double unused;
    const Cons<double> v = ReconFlux<P, RK, false>(L, R, T(0), T(0), pc, g, inv_gm1, &unused);
    f[dir][0][ty][tx] = v.d, f[dir][o1][ty][tx] = v.mx, f[dir][o2][ty][tx] = v.my, f[dir][o3][ty][tx] = v.mz;
    f[dir][4][ty][tx] = v.E;
  }
  __syncthreads();
  double m = 0.0;
  if (dir == 0 && tx >= 1 && tx < kS2X - 1 && ty >= 1 && ty < kS2Y - 1 && i < nx - ng && j < ny - ng) {
    const long id   = i + long(j) * nx;
    const double dt = dt_dev ? *dt_dev : dt_host, dtodx = dt / dx, dtody = dt / dy;
    double un[5];
#pragma unroll
    for (int q = 0; q < 5; q++)
      un[q] = U[q * nc + id] + (dtodx * (f[0][q][ty][tx - 1] - f[0][q][ty][tx]) +
                                dtody * (f[1][q][ty - 1][tx] - f[1][q][ty][tx]));
#pragma unroll
    for (int q = 0; q < 5; q++) U[q * nc + id] = un[q];
    const double d = un[0], dinv = 1.0 / d;
    const double vx = un[1] * dinv, vy = un[2] * dinv, vz = un[3] * dinv;
    const double pr = Fmax((un[4] - 0.5 * d * (vx * vx + vy * vy + vz * vz)) * (gamma - 1.0), 1.0e-20);
    const double cs = __builtin_sqrt(dinv * gamma * pr);
    m               = Fmax((Fabs(vx) + cs) / dx, (Fabs(vy) + cs) / dy);
    if (periodic) {  // every image of the cell in the ghost layers (each axis holds >= ng real cells)
      const int Lx = nx - 2 * ng, Ly = ny - 2 * ng;
      if (i < 2 * ng || i >= nx - 2 * ng || j < 2 * ng || j >= ny - 2 * ng)
        for (int b = -1; b <= 1; b++)
          for (int a = -1; a <= 1; a++) {
            const int gi = i + a * Lx, gj = j + b * Ly;
            if ((a | b) == 0 || gi < 0 || gi >= nx || gj < 0 || gj >= ny) continue;
#pragma unroll
            for (int q = 0; q < 5; q++) U[q * nc + gi + long(gj) * nx] = un[q];
          }
    }
  }
  if (dti) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = Fmax(m, __shfl_xor(m, off, 64));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    if (tid == 0) {
      double v = red[0];
      for (int q = 1; q < NT / 64; q++) v = Fmax(v, red[q]);
      atomicMax(dti, (unsigned long long)__double_as_longlong(v));
    }
  }
}

template <class P, int RK>
static hipError_t LaunchVl2dFusedP(double *U, double *W, int nx, int ny, int ng, double dx, double dy,
                                   const double *dt_dev, double dt, double gamma, bool periodic,
                                   unsigned long long *dti, hipStream_t s)
{
  auto tiles = [](int cells, int per) { return unsigned((cells + per - 1) / per); };
  hipLaunchKernelGGL((Vl2dStage1Kernel<P>), dim3(tiles(nx - 2, kS1X - 1), tiles(ny - 2, kS1Y - 1)), dim3(2 * kS1Cells),
                     0, s, U, W, nx, ny, dx, dy, dt_dev, dt, gamma, dti);
  hipLaunchKernelGGL((Vl2dStage2Kernel<P, RK>), dim3(tiles(nx - 2 * ng, kS2X - 2), tiles(ny - 2 * ng, kS2Y - 2)),
                     dim3(2 * kS2Cells), 0, s, U, W, nx, ny, ng, dx, dy, dt_dev, dt, gamma, int(periodic), dti);
  return hipGetLastError();
}

bool Vl2dFusedTakes(int ny, int recon, int riemann, bool de, const GravSpec &grav)
{
  return (recon == kPLMC || recon == kPPMC) && riemann == kRiemannHllc && !de && grav.id == 0 &&
         ny < 7 * 65535;  // the y tiles of one launch
}

hipError_t LaunchVl2dFused(double *U, double *W, int nx, int ny, int ng, int recon, int form, double dx, double dy,
                           const double *dt_dev, double dt, double gamma, bool periodic, unsigned long long *dti,
                           hipStream_t s)
{
  if (recon != kPLMC && recon != kPPMC) return hipErrorInvalidValue;
  CHL_SMALL_FORM(LaunchVl2dFusedP, U, W, nx, ny, ng, dx, dy, dt_dev, dt, gamma, periodic, dti, s);
}

}  // namespace chl
