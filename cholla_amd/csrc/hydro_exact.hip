// hydro_exact.hip -- PolicyExact instantiations of the fused VL kernels.
// Built with -ffp-contract=off: every product and sum rounds as the reference
// source writes it, so results match a strict IEEE restatement bit for bit.
#include "vl3d_launch.hpp"

namespace chl
{
hipError_t LaunchStage1Exact(const StepArgs &a, int R1, int tile, hipStream_t s)
{
  return LaunchStage1<PolicyExact>(a, R1, tile, s);
}
hipError_t LaunchStage2Exact(const StepArgs &a, int recon, int tile, hipStream_t s)
{
  return LaunchStage2<PolicyExact>(a, recon, tile, s);
}
hipError_t LaunchRepairExact(const StepArgs &a, hipStream_t s) { return LaunchRepair<PolicyExact>(a, s); }

// The side buffer of a density repair next to fused periodic images, one lane per face cell,
// and in a workgroup of its own the device clock (clk.dti null: no clock).  Neither reads what
// the other writes, and a launch of its own cost the clock its 1.4 us: a 64x32x32 step 55.6 ->
// 54.1 us (PLMC, reference order); this launch is the 3.9 us of its side buffer either way.
__global__ void RepairSideKernel(const double *U, double *side, int nx, int ny, int nz, int ng, StepClock clk)
{
  if (blockIdx.x + 1 == gridDim.x) {
    if (clk.dti && threadIdx.x == 0)
      AdvanceClock(__longlong_as_double((long long)*clk.dti), clk.dt, clk.t, clk.tout, clk.cfl, clk.nstep);
    return;
  }
  RepairSideCell(U, side, nx, ny, nz, ng, long(blockIdx.x) * blockDim.x + threadIdx.x);
}

hipError_t LaunchRepairSide(const StepArgs &a, const StepClock &clk, hipStream_t s)
{
  const long Lx = a.nx - 2 * a.ng, Ly = a.ny - 2 * a.ng, Lz = a.nz - 2 * a.ng;
  const long n  = 2 * (Ly * Lz + Lx * Lz + Lx * Ly);
  hipLaunchKernelGGL(RepairSideKernel, dim3(unsigned((n + 255) / 256 + 1)), dim3(256), 0, s, a.U, a.rep.side, a.nx,
                     a.ny, a.nz, a.ng, clk);
  return hipGetLastError();
}
}  // namespace chl
