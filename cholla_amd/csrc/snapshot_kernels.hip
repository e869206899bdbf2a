// snapshot_kernels.hip -- real cells of one field between Cholla's grid layout and the
// snapshot layout of its HDF5 files.
//
// The grid is x-fastest with ghost cells, id = i + j*nx + k*nx*ny; a snapshot dataset of
// real cells is z-fastest, buf = k + j*nz_real + i*nz_real*ny_real (CopyReal3D_GPU_Kernel,
// src/io/io_gpu.cu:44-60; Fill_HDF5_Buffer_From_Grid_CPU and Fill_Grid_From_HDF5_Buffer,
// src/io/io.cpp:1232-1268 and 2450-2490).  Between the two the fastest index changes from x
// to z, so each workgroup moves a tile of one y row through LDS, 64 (x) by 32 (z) or 32 by 32:
// the grid side reads (or writes) rows of consecutive x and the snapshot side writes (or reads)
// rows of 32 consecutive z.  Bound by HBM on large fields: 16 bytes per cell.  Grid rows start
// n_ghost cells into a line, so neighbouring tiles share a line at each row end; the 64 x 32
// tiles go out in XCD-contiguous order, x fastest, which keeps both halves of that line in one
// L2 (two XCDs each fetched it, or wrote its half through).  Launched over and over, a 256^3
// field: unpack 84.7 -> 61.9 us, pack 54.7 -> 54.8; 300x212x190: pack 57.8 -> 42.4 us, unpack 56.4
// -> 44.0 (4.3-4.9 TB/s; a plain copy reaches 4.8), against 32x32 tiles in dispatch order.  In
// passes of five packs and five unpacks of a 256^3 state they take 73 and 52 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>

#include "snapshot_kernels.hpp"

namespace chl
{
namespace
{

constexpr int kTZ = 32;  // tile: TX by kTZ, x by z
constexpr int kThreads = 256;

// PACK: grid -> buf (converted to OUT); !PACK: buf -> grid.  (ox, oy, oz) is the grid index of
// the dataset's first element: n_ghost, or n_ghost - 1 along a magnetic field's own axis
// (its dataset holds one more face than there are real cells).  TX 64: a linear grid of
// the tiles from `first` on in XCD-contiguous order; TX 32: the grid's axes are the tiles'.
template <bool PACK, typename OUT, int kTX>
__global__ void __launch_bounds__(kThreads) SnapshotTileKernel(double *grid, OUT *buf, int nx, int ny, int nxr, int nyr,
                                                              int nzr, int ox, int oy, int oz, unsigned gx,
                                                              unsigned gz, unsigned first, unsigned tiles)
{
  __shared__ double t[kTZ][kTX + 1];
  int i0, k0, j;
  if constexpr (kTX == 64) {
    const unsigned per = (tiles + 7) / 8, n = (blockIdx.x & 7) * per + (blockIdx.x >> 3), q = first + n;
    if ((blockIdx.x >> 3) >= per || n >= tiles) return;
    i0 = int(q % gx) * kTX, k0 = int(q / gx % gz) * kTZ, j = int(q / (gx * gz));
  } else {
    i0 = int(blockIdx.x) * kTX, k0 = int(blockIdx.y) * kTZ, j = int(blockIdx.z);
  }
  const size_t plane = size_t(nx) * ny;
  auto gid = [&](int i, int k) { return size_t(i + ox) + size_t(j + oy) * nx + size_t(k + oz) * plane; };
  auto bid = [&](int i, int k) { return size_t(k) + size_t(j) * nzr + size_t(i) * nzr * nyr; };
  const int ax = threadIdx.x % kTX, az = threadIdx.x / kTX;  // grid rows: consecutive x
  const int bz = threadIdx.x % kTZ, bx = threadIdx.x / kTZ;  // snapshot rows: consecutive z
  if constexpr (PACK) {
#pragma unroll
    for (int kk = az; kk < kTZ; kk += kThreads / kTX) {
      const int i = i0 + ax, k = k0 + kk;
      if (i < nxr && k < nzr) t[kk][ax] = grid[gid(i, k)];
    }
    __syncthreads();
#pragma unroll
    for (int ii = bx; ii < kTX; ii += kThreads / kTZ) {
      const int i = i0 + ii, k = k0 + bz;
      if (i < nxr && k < nzr) buf[bid(i, k)] = OUT(t[bz][ii]);
    }
  } else {
#pragma unroll
    for (int ii = bx; ii < kTX; ii += kThreads / kTZ) {
      const int i = i0 + ii, k = k0 + bz;
      if (i < nxr && k < nzr) t[bz][ii] = double(buf[bid(i, k)]);
    }
    __syncthreads();
#pragma unroll
    for (int kk = az; kk < kTZ; kk += kThreads / kTX) {
      const int i = i0 + ax, k = k0 + kk;
      if (i < nxr && k < nzr) grid[gid(i, k)] = t[kk][ax];
    }
  }
}

// From this many cells the tiles are 64 x 32 in XCD-contiguous order.  Below it a field and its
// buffer stay in the caches, lines shared by two XCDs cost little and more, smaller workgroups
// start sooner: 10 transposes and their launches of 80^3 take 166 us in 32 x 32 tiles against
// 182, 160^3 308 against 313, 200^3 456 against 454, 256^3 841 against 748.
constexpr size_t kLargeField = size_t(8) << 20;

template <bool PACK, typename OUT>
hipError_t Launch(double *grid, OUT *buf, const SnapshotShape &s, hipStream_t st)
{
  const unsigned gz = unsigned((s.nzr + kTZ - 1) / kTZ);
  if (size_t(s.nxr) * s.nyr * s.nzr < kLargeField && s.nyr <= 65535) {
    hipLaunchKernelGGL((SnapshotTileKernel<PACK, OUT, 32>), dim3(unsigned((s.nxr + 31) / 32), gz, unsigned(s.nyr)),
                       dim3(kThreads), 0, st, grid, buf, s.nx, s.ny, s.nxr, s.nyr, s.nzr, s.ox, s.oy, s.oz, 0u, 0u, 0u,
                       0u);
    return hipGetLastError();
  }
  // 2^23 tiles a launch: one of 2^24 has the 2^32 threads that a launch may not reach, which a 2D
  // field of 32768^2 does
  constexpr size_t kPerLaunch = size_t(1) << 23;
  const unsigned gx = unsigned((s.nxr + 63) / 64);
  const size_t all  = size_t(gx) * gz * s.nyr;
  for (size_t first = 0; first < all; first += kPerLaunch) {
    const unsigned tiles = unsigned(std::min(kPerLaunch, all - first));
    hipLaunchKernelGGL((SnapshotTileKernel<PACK, OUT, 64>), dim3((tiles + 7) / 8 * 8), dim3(kThreads), 0, st, grid,
                       buf, s.nx, s.ny, s.nxr, s.nyr, s.nzr, s.ox, s.oy, s.oz, gx, gz, unsigned(first), tiles);
    if (const hipError_t e = hipGetLastError()) return e;
  }
  return hipSuccess;
}

}  // namespace

hipError_t LaunchSnapshotPack(const double *grid, double *buf, const SnapshotShape &s, hipStream_t st)
{
  return Launch<true, double>(const_cast<double *>(grid), buf, s, st);
}

hipError_t LaunchSnapshotPack32(const double *grid, float *buf, const SnapshotShape &s, hipStream_t st)
{
  return Launch<true, float>(const_cast<double *>(grid), buf, s, st);
}

hipError_t LaunchSnapshotUnpack(const double *buf, double *grid, const SnapshotShape &s, hipStream_t st)
{
  return Launch<false, double>(grid, const_cast<double *>(buf), s, st);
}

}  // namespace chl
