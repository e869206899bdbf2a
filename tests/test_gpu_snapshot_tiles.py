"""The snapshot transposes at the edges of their tiles (32 x 32, and 64 x 32 from 2^23 cells on),
against the numpy transpose."""
import numpy as np
import pytest

import cholla_amd as chl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("direction", [-1, 0, 1, 2])
@pytest.mark.parametrize("dims", [(1, 2, 1), (63, 3, 31), (64, 2, 32), (65, 5, 33), (9, 1, 130), (200, 7, 4)])
def test_pack_and_unpack_tiles(dims, direction):
    nxr, nyr, nzr = dims
    ng = 3
    nx, ny, nz = nxr + 2 * ng, nyr + 2 * ng, nzr + 2 * ng
    ext = [n + (direction == a) for a, n in enumerate(dims)]
    lo = [ng - (direction == a) for a in range(3)]
    rng = np.random.default_rng(1)
    F = rng.normal(size=(nz, ny, nx))
    want = F[lo[2]:lo[2] + ext[2], lo[1]:lo[1] + ext[1], lo[0]:lo[0] + ext[0]].transpose(2, 1, 0)
    D, buf = chl.DeviceArray.from_host(F), chl.DeviceArray(want.size, np.full(want.size, -7.0))
    args = (nx, ny, nz, ng, *ext, direction)
    chl.check(chl.lib().chl_pack_real_cells(D.ptr, buf.ptr, *args))
    assert np.array_equal(buf.download().reshape(want.shape), want)
    b32 = chl.DeviceArray(want.size, np.zeros(want.size))
    chl.check(chl.lib().chl_pack_real_cells_f32(D.ptr, b32.ptr, *args))
    assert np.array_equal(b32.download().view(np.float32)[:want.size].reshape(want.shape), want.astype(np.float32))
    G0 = rng.normal(size=F.shape)
    G = chl.DeviceArray.from_host(G0)
    chl.check(chl.lib().chl_unpack_real_cells(buf.ptr, G.ptr, *args))
    out = G0.copy()
    out[lo[2]:lo[2] + ext[2], lo[1]:lo[1] + ext[1], lo[0]:lo[0] + ext[0]] = want.transpose(2, 1, 0)
    assert np.array_equal(G.download().reshape(F.shape), out)


@pytest.mark.parametrize("dims", [(65, 3, 43019), (8388607, 1, 1), (129, 2033, 32), (64, 4096, 33)])
def test_pack_and_unpack_large_fields(dims):
    # just below and above the size where the tiles change, with remainders in x and z
    rng = np.random.default_rng(2)
    F = rng.normal(size=dims[::-1])
    want = F.transpose(2, 1, 0)
    D, buf = chl.DeviceArray.from_host(F), chl.DeviceArray(F.size, np.zeros(F.size))
    args = (*dims, 0, *dims, -1)
    chl.check(chl.lib().chl_pack_real_cells(D.ptr, buf.ptr, *args))
    assert np.array_equal(buf.download().reshape(want.shape), want)
    G = chl.DeviceArray(F.size, np.zeros(F.size))
    chl.check(chl.lib().chl_unpack_real_cells(buf.ptr, G.ptr, *args))
    assert np.array_equal(G.download().reshape(F.shape), F)


def test_more_tiles_than_one_launch_holds():
    """2^24 tiles of 256 threads exceed a launch: 258 tiles along z of 65535 one-cell-wide rows, 4.3 GB."""
    ny, nz = 65535, 8225
    F = np.arange(ny * nz, dtype=np.float64)
    D, buf = chl.DeviceArray.from_host(F), chl.DeviceArray(F.size)
    args = (1, ny, nz, 0, 1, ny, nz, -1)
    chl.check(chl.lib().chl_pack_real_cells(D.ptr, buf.ptr, *args))
    got = buf.download().reshape(ny, nz)
    rows = np.r_[0:3, 3:ny - 3:509, ny - 3:ny]  # every launch's share, first and last rows whole
    want = np.arange(nz, dtype=np.float64)[None, :] * ny + rows[:, None]
    assert np.array_equal(got[rows], want)
    del got
    chl.check(chl.lib().chl_memcpy_dtod(D.ptr, buf.ptr, 8))  # spoil one element, then unpack over it
    chl.check(chl.lib().chl_unpack_real_cells(buf.ptr, D.ptr, *args))
    assert np.array_equal(D.download(), F)
