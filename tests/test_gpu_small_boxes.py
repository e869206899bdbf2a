"""The fused 1D and 2D steps (vl_small.hip) against the CPU oracle: bit-identical in the
reference-order form at the sizes where the one-workgroup line and the 2D tiles begin, end and
leave remainders, for every boundary; the other forms within their bars."""
import numpy as np
import pytest

import cholla_amd as chl
from helpers import check_fp64, check_mixed, interior, rel_l1
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
RECON = {orc.PLMC: chl.RECON_PLMC, orc.PPMC: chl.RECON_PPMC}


def wave_line(n_real, ng, gamma, seed=2):
    n = n_real + 2 * ng
    rng = np.random.default_rng(seed)
    x = (np.arange(n) - ng + 0.5) / n_real
    d = np.where(x < 0.5, 1.0, 0.3) + 0.05 * rng.uniform(-1, 1, n)
    v = [0.3 * np.sin(2 * np.pi * x), 0.1 * rng.uniform(-1, 1, n), 0.2 * np.cos(2 * np.pi * x)]
    p = np.where(x < 0.5, 1.0, 0.2)
    U = np.stack([d, d * v[0], d * v[1], d * v[2], p / (gamma - 1) + 0.5 * d * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)])
    return U.reshape(-1).copy(), n


# one wave; a full and a just over-full workgroup; two cells a thread; the last fused size and the
# first that is not (n counts the 4 ghost cells on each side)
@pytest.mark.parametrize("n_real", [4, 56, 57, 503, 504, 505, 1015, 1016, 1017])
@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("bc", [(1, 1), (3, 3), (2, 3)])
def test_line_batch_bitwise(n_real, recon, bc):
    ng, g = 4, 1.4
    U, n = wave_line(n_real, ng, g)
    flags = [*bc, 0, 0, 0, 0]
    orc.set_boundaries(U, n, 1, 1, 5, ng, flags)
    h = 1.0 / n_real
    A = U.copy()
    steps_o, t_o = orc.run(A, n, 1, 1, ng, 5, h, h, h, g, recon, flags, 0.25, 1e30, 5)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(n, 1, 1, ng, RECON[recon], chl.PREC_FP64_EXACT, bc=[*bc, 1, 1, 1, 1])
    steps, t = hy.run(D, h, h, h, g, 0.25, 1e30, 5)
    assert (steps, t) == (steps_o, t_o) and np.array_equal(D.download(), A)


def test_line_batch_stops_at_the_output_time():
    # the last step is clamped to tout, later ones change nothing, and a second call goes on
    ng, g = 4, 1.4
    U, n = wave_line(80, ng, g)
    flags = [3, 3, 0, 0, 0, 0]
    orc.set_boundaries(U, n, 1, 1, 5, ng, flags)
    h = 1.0 / 80
    A = U.copy()
    so, to = orc.run(A, n, 1, 1, ng, 5, h, h, h, g, orc.PLMC, flags, 0.0, 0.02, 5000)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(n, 1, 1, ng, chl.RECON_PLMC, chl.PREC_FP64_EXACT, bc=[3, 3, 1, 1, 1, 1])
    s, t = hy.run(D, h, h, h, g, 0.0, 0.02, 5000)
    assert (s, t) == (so, to) and t == 0.02 and np.array_equal(D.download(), A)
    assert hy.run(D, h, h, h, g, 0.02, 0.02, 10) == (0, 0.02)
    assert np.array_equal(D.download(), A)
    # more steps than one launch carries
    so, to = orc.run(A, n, 1, 1, ng, 5, h, h, h, g, orc.PLMC, flags, 0.02, 1e30, 1500)
    assert hy.run(D, h, h, h, g, 0.02, 1e30, 1500) == (so, to)
    assert np.array_equal(D.download(), A)
    ms, dt = hy.time_steps(D, h, h, h, g, 1030)
    orc.run(A, n, 1, 1, ng, 5, h, h, h, g, orc.PLMC, flags, 0.0, 1e300, 1030)
    assert np.array_equal(D.download(), A) and dt > 0


def wave_plane(nx_real, ny_real, ng, gamma, seed=3):
    nx, ny = nx_real + 2 * ng, ny_real + 2 * ng
    rng = np.random.default_rng(seed)
    X, Y = np.meshgrid((np.arange(nx) - ng + 0.5) / nx_real, (np.arange(ny) - ng + 0.5) / ny_real)
    d = np.where(np.abs(Y - 0.5) < 0.25, 2.0, 1.0) + 0.1 * np.sin(2 * np.pi * X)
    v = [0.5 * np.cos(2 * np.pi * Y), 0.2 * np.sin(4 * np.pi * X), 0.1 * rng.uniform(-1, 1, X.shape)]
    p = 2.5 + 0.3 * rng.uniform(-1, 1, X.shape)
    U = np.stack([d, d * v[0], d * v[1], d * v[2], p / (gamma - 1) + 0.5 * d * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)])
    return U.reshape(-1).copy(), nx, ny


# a box inside one tile (stage 2 updates 30 x 10, stage 1 31 x 7), tiles met exactly, remainders
@pytest.mark.parametrize("dims", [(4, 5), (30, 10), (31, 11), (23, 41), (61, 20), (90, 33)])
@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("bc", [(1, 1, 1, 1), (3, 2, 1, 1), (2, 2, 3, 3)])
@pytest.mark.parametrize("use_graph", [False, True])
def test_plane_step_bitwise(dims, recon, bc, use_graph):
    ng, g = 4, 5 / 3
    U, nx, ny = wave_plane(*dims, ng, g)
    flags = [*bc, 0, 0]
    orc.set_boundaries(U, nx, ny, 1, 5, ng, flags)
    w = (1.0 / dims[0], 1.3 / dims[1], 1.0)
    A = U.copy()
    so, to = orc.run(A, nx, ny, 1, ng, 5, *w, g, recon, flags, 0.0, 1e30, 4)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(nx, ny, 1, ng, RECON[recon], chl.PREC_FP64_EXACT, bc=[*bc, 1, 1])
    s, t = hy.run(D, *w, g, 0.0, 1e30, 4, use_graph=use_graph)
    assert (s, t) == (so, to) and np.array_equal(D.download(), A)


@pytest.mark.parametrize("precision", [chl.PREC_FP64, chl.PREC_MIXED])
@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
def test_other_forms_within_their_bars(recon, precision):
    ng, check = 4, check_fp64 if precision == chl.PREC_FP64 else check_mixed
    U, n = wave_line(300, ng, 1.4)
    flags = [1, 1, 0, 0, 0, 0]
    orc.set_boundaries(U, n, 1, 1, 5, ng, flags)
    A, D = U.copy(), chl.DeviceArray.from_host(U)
    orc.run(A, n, 1, 1, ng, 5, 1 / 300, 1, 1, 1.4, recon, flags, 0.0, 1e30, 4)
    chl.Hydro(n, 1, 1, ng, RECON[recon], precision).run(D, 1 / 300, 1, 1, 1.4, 0.0, 1e30, 4)
    check([rel_l1(a, b) for a, b in zip(interior(D.download(), 5, 1, 1, n, ng), interior(A, 5, 1, 1, n, ng))])
    U, nx, ny = wave_plane(45, 37, ng, 5 / 3)
    flags = [1, 1, 1, 1, 0, 0]
    orc.set_boundaries(U, nx, ny, 1, 5, ng, flags)
    A, D = U.copy(), chl.DeviceArray.from_host(U)
    orc.run(A, nx, ny, 1, ng, 5, 1 / 45, 1 / 37, 1, 5 / 3, recon, flags, 0.0, 1e30, 4)
    chl.Hydro(nx, ny, 1, ng, RECON[recon], precision).run(D, 1 / 45, 1 / 37, 1, 5 / 3, 0.0, 1e30, 4)
    check([rel_l1(a, b) for a, b in zip(interior(D.download(), 5, 1, ny, nx, ng), interior(A, 5, 1, ny, nx, ng))])
