// mhd_launch.hpp -- host dispatch of the MHD step kernels.
#pragma once

#include <algorithm>
#include <cmath>

#include "mhd_kernels.hpp"
#include "support_kernels.hpp"

namespace chl
{

inline unsigned MhdBlocks(size_t n) { return unsigned((n + 255) / 256); }

// Planes per workgroup of a launch whose workgroups march: `columns` of them per chunk over
// `planes` planes, with `slots` running at a time.  The least rounds x (k + c0), c0 the planes'
// worth of work a chunk starts with (its prologue), up to cap (where longer chunks measured
// slower on Orszag-Tang 256^3).  Chunks of 16 on every box left a 56x40x36 one to 18-54
// workgroups: its CT updates and y / z fluxes took 79-97 us each (reference order), and its
// step 400 us against 125.
inline int MhdChunk(long columns, int planes, int slots, double c0, int cap)
{
  double best = 1e300;
  int pick    = 1;
  for (int k : {1, 2, 3, 4, 6, 8, 12, 16}) {
    if (k > cap) break;
    const double groups = double(columns) * ((planes + k - 1) / k);
    const double rounds = groups <= 4.0 * slots ? std::ceil(groups / slots) : groups / slots + 0.5;
    const double cost   = rounds * (k + c0);
    if (cost < best) best = cost, pick = k;
  }
  return pick;
}

// The three stage-2 flux launches of a reconstruction RK (1 PLMC, 2 PPMC) over the faces
// with every index in [lo, hi], in XCD-contiguous order: x faces in 64 x 4 face tiles, y and
// z faces in 64 x 4 columns that march along the direction (MhdChunk).
template <class P, int RK>
void MhdFlux2Tiles(const mhd::MhdArgs &a, int lo, int hx, int hy, int hz, hipStream_t s)
{
  const unsigned ex = unsigned(hx - lo + 1), ey = unsigned(hy - lo + 1), ez = unsigned(hz - lo + 1);
  auto blocks = [](unsigned t) { return dim3((t + 7) / 8 * 8); };
  // counted as two workgroups per CU in the mixed form and one in FP64, fewer than the registers
  // admit (3-4 and 1-2).  The chunk so taken costs a step up to 4 % against the best one (64^3,
  // mixed), under 1 % from 128^3 on
  constexpr int kSlots = P::kId == PolicyMixed::kId ? 512 : 256;
  const unsigned bx = (ex + 63) / 64;
  const unsigned ky = unsigned(MhdChunk(long(bx) * ((ez + 3) / 4), int(ey), kSlots, 1.0, 16));
  const unsigned kz = unsigned(MhdChunk(long(bx) * ((ey + 3) / 4), int(ez), kSlots, 1.0, 16));
  hipLaunchKernelGGL((mhd::MhdFlux2TileKernel<P, RK>), blocks((ex + 63) / 64 * ((ey + 3) / 4) * ez), dim3(256), 0,
                     s, a, lo, hx, hy, hz);
  hipLaunchKernelGGL((mhd::MhdFlux2MarchKernel<P, 1, RK>), blocks(bx * ((ez + 3) / 4) * ((ey + ky - 1) / ky)),
                     dim3(256), 0, s, a, lo, hx, hy, hz, int(ky));
  hipLaunchKernelGGL((mhd::MhdFlux2MarchKernel<P, 2, RK>), blocks(bx * ((ey + 3) / 4) * ((ez + kz - 1) / kz)),
                     dim3(256), 0, s, a, lo, hx, hy, hz, int(kz));
}

// The tiles of the CT-update launches, and their planes per workgroup: as many workgroups run on
// a CU as their LDS admits, three of the mixed form (48 KB of 160) and two of the FP64 ones
// (72 KB).  Counted as three, these took 12 planes where 16 are faster: Orszag-Tang 128^3 in
// FP64, the full update 241 us against 206.
constexpr int kCtX = 32, kCtY = 8;
template <class P>
int MhdCtChunk(long columns, int planes)
{
  constexpr size_t lds = 2 * sizeof(mhd::CtPlane<typename P::T, kCtX + 2, kCtY + 2>) +
                         3 * (kCtX + 1) * (kCtY + 1) * sizeof(double);
  constexpr int per_cu = lds <= 160 * 1024 / 3 ? 3 : 2;
  static_assert(per_cu * lds <= 160 * 1024, "the workgroups of a CU share its LDS");
  return MhdChunk(columns, planes, 256 * per_cu, 1.5, 16);
}

// CT edge fields fused with one stage's update (MhdCtUpdateKernel) over the cells [clo, ch*]
// and the edges [elo, eh*]: 32 x 8 tiles, z-chunks of up to 16 planes (on Orszag-Tang 256^3
// these ran 2-5 % faster than 16 x 16 tiles or z-chunks of 8 and 32).  Over boxes of 32^3 to
// 256^3 the chunk taken costs a step 0.05 % in the mean against the best of all, 1.1 % at worst.
template <class P, bool FULL>
void MhdCtUpdate(const mhd::MhdArgs &a, int clo, int chx, int chy, int chz, int elo, int ehx, int ehy, int ehz,
                 hipStream_t s)
{
  constexpr int CTX = kCtX, CTY = kCtY;
  const int columns    = ((chx - clo + CTX) / CTX) * ((chy - clo + CTY) / CTY);
  const int kchunk     = MhdCtChunk<P>(columns, chz - clo + 1);
  const unsigned tiles = unsigned(columns * ((chz - clo + kchunk) / kchunk));
  hipLaunchKernelGGL((mhd::MhdCtUpdateKernel<P, CTX, CTY, FULL>), dim3((tiles + 7) / 8 * 8), dim3(CTX * CTY), 0, s, a,
                     clo, chx, chy, chz, elo, ehx, ehy, ehz, kchunk);
}

// One VL step of MHD: stage-1 fluxes, edge fields + half update, stage-2 fluxes, edge
// fields + full update.  The ghost refresh is a separate launch; the inverse-dt reduction is
// folded into the stage-1 flux launch (kFlagFoldDt, device clock advanced right after it)
// or left to MhdCalcDtKernel.
template <class P>
hipError_t MhdStepT(const mhd::MhdArgs &a, hipStream_t s)
{
  const int nx = a.nx, ny = a.ny, nz = a.nz, ng = a.ng;
  // stage-1 faces i+1/2 of every cell with i <= n-2 (other indices over the whole grid)
  const mhd::MhdRegion m1 = mhd::MakeMhdSlab(0, nx - 1, ny - 1, nz - 1);
  if constexpr (P::kId == PolicyMixed::kId) {
    // z-march in 32 x 8 tiles of up to 8 planes (OT 256^3: 0.98 ms against 1.02 for the per-cell
    // launch; the FP64 forms run slower there, at 2 waves per SIMD against 3)
    constexpr int TX = 32, TY = 8;
    const int columns     = ((nx + TX - 1) / TX) * ((ny + TY - 1) / TY);
    const int kz          = MhdChunk(columns, nz, 1024, 0.7, 8);  // four workgroups per CU
    const unsigned blocks = unsigned(columns * ((nz + kz - 1) / kz));
    hipLaunchKernelGGL((mhd::MhdFlux1MarchKernel<P, TX, TY>), dim3((blocks + 7) / 8 * 8), dim3(TX * TY), 0, s, a, kz);
  } else {
    hipLaunchKernelGGL((mhd::MhdFlux1AllKernel<P>), dim3(mhd::MhdRegionBlocks(m1)), dim3(256), 0, s, a, m1);
  }
  if (a.flags & kFlagFoldDt) {
    const hipError_t e = LaunchDtAdvance(a.dti, a.clk_dt, a.clk_t, a.clk_tout, a.clk_cfl, a.clk_nstep, s, true);
    if (e != hipSuccess) return e;
  }
  // edges [2, n-1], half update of the cells [1, n-2]
  MhdCtUpdate<P, false>(a, 1, nx - 2, ny - 2, nz - 2, 2, nx - 1, ny - 1, nz - 1, s);
  {  // stage-2 faces with every index in [ng - 1, n - ng]
    const int lo = ng - 1, hx = nx - ng, hy = ny - ng, hz = nz - ng;
    if (a.recon == 0) {
      const mhd::MhdRegion m2 = mhd::MakeMhdSlab(lo, hx, hy, hz);
      hipLaunchKernelGGL((mhd::MhdFlux2PcmKernel<P>), dim3(mhd::MhdRegionBlocks(m2)), dim3(256), 0, s, a, m2);
    } else if (a.recon == 2) {
      MhdFlux2Tiles<P, 2>(a, lo, hx, hy, hz, s);
    } else {
      MhdFlux2Tiles<P, 1>(a, lo, hx, hy, hz, s);
    }
  }
  // edges [ng, n-ng], full update of the real cells and of the face fields just below them
  MhdCtUpdate<P, true>(a, ng, nx - ng - 1, ny - ng - 1, nz - ng - 1, ng, nx - ng, ny - ng, nz - ng, s);
  return hipGetLastError();
}

hipError_t LaunchMhdStepExact(const mhd::MhdArgs &a, hipStream_t s);

}  // namespace chl
