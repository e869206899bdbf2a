"""HLLC faces of the forms that select one side's star state (hydro_physics.hpp: Hllc) in every
case of the selection: supersonic to the left and to the right, subsonic with the contact on
either side, colliding and receding streams, a stationary contact."""
import numpy as np
import pytest

import cholla_amd as chl
from helpers import FIELD_NAMES, check_fp64, check_mixed, interior, rel_l1
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
G, NG, DIMS = 5 / 3, 4, (40, 7, 6)
STREAMS = [((1, 3, 1), (0.5, 3, 0.4)), ((1, -3, 1), (0.5, -3, 0.4)), ((1, 0.4, 1), (0.3, 0.4, 0.9)),
           ((1, -0.4, 1), (0.3, -0.4, 0.9)), ((1, 1.5, 1), (1, -1.5, 1)), ((1, -0.5, 1), (1, 0.5, 1))]
RECON = {orc.PLMC: chl.RECON_PLMC, orc.PPMC: chl.RECON_PPMC}


def halves(left, right, noise, seed=9):
    """A periodic box whose two halves along x hold (d, vx, p), with noise (no two cells alike)."""
    nx, ny, nz = (v + 2 * NG for v in DIMS)
    rng = np.random.default_rng(seed)
    in_l = ((np.arange(nx) - NG) % DIMS[0] < DIMS[0] // 2)[None, None, :]
    d, vx, p = (np.where(in_l, a, b) * (1 + noise * rng.uniform(-1, 1, (nz, ny, nx))) for a, b in zip(left, right))
    vy, vz = noise * rng.uniform(-1, 1, (2, nz, ny, nx))
    U = np.stack([d, d * vx, d * vy, d * vz, p / (G - 1) + 0.5 * d * (vx ** 2 + vy ** 2 + vz ** 2)])
    U = U.reshape(-1).copy()
    orc.set_boundaries(U, nx, ny, nz, 5, NG, [1] * 6)
    return U, (nx, ny, nz)


def step(U, dims, recon, precision, steps, dual_energy=False):
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(*dims, NG, RECON[recon], precision, dual_energy=dual_energy)
    hy.run(D, *[1.0 / v for v in DIMS], G, 0.0, 1e30, steps)
    return D.download()


@pytest.mark.parametrize("precision", [chl.PREC_FP64, chl.PREC_MIXED])
@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("left,right", STREAMS)
def test_every_selection_within_the_forms_bars(left, right, recon, precision):
    U, dims = halves(left, right, 0.05)
    A = U.copy()
    orc.run(A, *dims, NG, 5, *[1.0 / v for v in DIMS], G, recon, [1] * 6, 0.0, 1e30, 2)
    B = step(U, dims, recon, precision, 2)
    l1 = [rel_l1(b, a) for b, a in zip(interior(B, 5, *dims, NG), interior(A, 5, *dims, NG))]
    (check_fp64 if precision == chl.PREC_FP64 else check_mixed)(l1)


@pytest.mark.parametrize("precision", [chl.PREC_FP64, chl.PREC_MIXED])
@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("left,right", STREAMS)
def test_dual_energy_faces_within_the_forms_bars(left, right, recon, precision):
    """The GasEnergy flux of each selection, with the gas energy well above the switch's 1e-3 of the
    total (the supersonic streams' internal energy is 5-30 % of it), so that no cell changes side."""
    U, dims = halves(left, right, 0.05)
    q = U.reshape(5, -1)
    U = np.concatenate([U, q[4] - 0.5 * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2) / q[0]])
    A = U.copy()
    orc.run(A, *dims, NG, 6, *[1.0 / v for v in DIMS], G, recon, [1] * 6, 0.0, 1e30, 2, dual_energy_on=True)
    B = step(U, dims, recon, precision, 2, dual_energy=True)
    l1 = [rel_l1(b, a) for b, a in zip(interior(B, 6, *dims, NG), interior(A, 6, *dims, NG))]
    names = tuple(FIELD_NAMES[:5]) + ("GasEnergy",)
    (check_fp64 if precision == chl.PREC_FP64 else check_mixed)(l1, names=names)


@pytest.mark.parametrize("precision", [chl.PREC_FP64, chl.PREC_MIXED])
@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
def test_stationary_contact_stays(recon, precision):
    U, dims = halves((1, 0, 1), (0.125, 0, 1), 0.0)
    assert np.array_equal(step(U, dims, recon, precision, 3), U)
