"""The FP64 quotients and square roots of the reference-order form over the exponent range.

The kernels divide without the compiler's range scaling (hydro_physics.hpp: Quot,
SqrtUnscaled), which has IEEE division's bits for numerators of at least 2^-969, and in full where
a numerator is a product of two slopes.  States whose density, pressure and transverse velocity
sit far from 1 (above the scheme's own floors of 1e-20) must therefore stay bit-identical to the
CPU oracle, in hydro of one, two and three dimensions with and without dual energy and in MHD.
The FP64 form's limiter takes a subnormal second difference as round-off."""
import numpy as np
import pytest

import cholla_amd as chl
from helpers import check_mixed, interior, rel_l1
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def scaled_box(n, ng, d_scale, p_scale, vz, gamma=5 / 3, seed=11):
    """A smooth periodic box with a density jump, in units d_scale and p_scale, with a third
    velocity component of size vz (in units of the sound speed)."""
    N = n + 2 * ng
    rng = np.random.default_rng(seed)
    x = (np.arange(N) - ng + 0.5) / n
    X, Y = x[None, None, :], x[None, :, None]
    d = np.where(np.abs(Y - 0.5) < 0.25, 2.0, 1.0) * (1 + 0.1 * np.sin(2 * np.pi * X)) + np.zeros((N, N, N))
    u = np.sqrt(p_scale / d_scale)
    v = [u * (np.where(np.abs(Y - 0.5) < 0.25, 0.5, -0.5) + 0 * d), u * 0.1 * np.sin(4 * np.pi * X) + 0 * d,
         u * vz * rng.uniform(-1, 1, (N, N, N))]
    d = d * d_scale
    E = 2.5 * p_scale / (gamma - 1) + 0.5 * d * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
    U = np.stack([d, d * v[0], d * v[1], d * v[2], E]).reshape(-1).copy()
    orc.set_boundaries(U, N, N, N, 5, ng, [1] * 6)
    return U, N


# vz of 1e-150 and 1e-158: products of two of its slopes are below 2^-969 and subnormal
SCALES = [(1.0, 1.0, 1e-280), (1.0, 1.0, 1e-150), (1.0, 1.0, 1e-158), (1.0, 2.0 ** 300, 1e-30),
          (2.0 ** 120, 2.0 ** 100, 1e-120), (2.0 ** 200, 2.0 ** -40, 0.0)]
RECON = {orc.PLMC: chl.RECON_PLMC, orc.PPMC: chl.RECON_PPMC, orc.PLMP: chl.RECON_PLMP, orc.PPMP: chl.RECON_PPMP}


@pytest.mark.parametrize("recon", list(RECON))
@pytest.mark.parametrize("d_scale,p_scale,vz", SCALES)
def test_exact_form_bitwise_far_from_one(recon, d_scale, p_scale, vz):
    n, ng, g = 16, 4, 5 / 3
    U, N = scaled_box(n, ng, d_scale, p_scale, vz)
    h = 1.0 / n
    A = U.copy()
    orc.run(A, N, N, N, ng, 5, h, h, h, g, recon, [1] * 6, 0.0, 1e300, 3)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(N, N, N, ng, RECON[recon], chl.PREC_FP64_EXACT)
    hy.run(D, h, h, h, g, 0.0, 1e300, 3)
    assert np.isfinite(A).all()
    assert np.array_equal(D.download(), A)


@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("solver", [orc.HLLC, orc.ROE])  # HLLC: the batched 1D and fused 2D steps
@pytest.mark.parametrize("two_d", [False, True])
@pytest.mark.parametrize("d_scale,p_scale,vz", SCALES)
def test_exact_form_bitwise_far_from_one_1d_2d(two_d, solver, recon, d_scale, p_scale, vz):
    n, ng, g = 16, 4, 5 / 3
    U, N = scaled_box(n, ng, d_scale, p_scale, vz)
    box = U.reshape(5, N, N, N)
    U = (box[:, N // 2] if two_d else box[:, N // 2, N // 2]).reshape(-1).copy()
    dims = (N, N, 1) if two_d else (N, 1, 1)
    flags = [1] * 4 + [0] * 2 if two_d else [1] * 2 + [0] * 4
    h = 1.0 / n
    A = U.copy()
    orc.run(A, *dims, ng, 5, h, h, h, g, recon, flags, 0.0, 1e300, 3, solver=solver)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(*dims, ng, RECON[recon], chl.PREC_FP64_EXACT,
                   riemann={orc.HLLC: chl.RIEMANN_HLLC, orc.ROE: chl.RIEMANN_ROE}[solver])
    hy.run(D, h, h, h, g, 0.0, 1e300, 3)
    # (Roe's averages overflow at the last scale, in the oracle too)
    assert np.isfinite(A).all() or solver == orc.ROE
    assert np.array_equal(D.download(), A, equal_nan=True)


@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("d_scale,p_scale,vz", SCALES)
def test_exact_form_bitwise_far_from_one_dual_energy(recon, d_scale, p_scale, vz):
    n, ng, g = 16, 4, 5 / 3
    U, N = scaled_box(n, ng, d_scale, p_scale, vz)
    q = U.reshape(5, -1)
    U = np.concatenate([U, q[4] - 0.5 * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2) / q[0]])
    h = 1.0 / n
    A = U.copy()
    orc.run(A, N, N, N, ng, 6, h, h, h, g, recon, [1] * 6, 0.0, 1e300, 3, dual_energy_on=True)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(N, N, N, ng, RECON[recon], chl.PREC_FP64_EXACT, dual_energy=True)
    hy.run(D, h, h, h, g, 0.0, 1e300, 3)
    assert np.isfinite(A).all()
    assert np.array_equal(D.download(), A)


@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("d_scale,p_scale,vz", SCALES)
def test_exact_form_bitwise_far_from_one_mhd(recon, d_scale, p_scale, vz):
    """Uniform B along x and y (divergence-free) of the pressure's scale, and a Bz of vz's."""
    n, ng, g = 16, 5, 5 / 3
    U, N = scaled_box(n, ng, d_scale, p_scale, vz)
    one = np.ones(N ** 3)
    bx, by, bz = 0.3 * np.sqrt(p_scale), 0.2 * np.sqrt(p_scale), np.sqrt(p_scale) * vz
    U = np.concatenate([U, bx * one, by * one, bz * one])
    U.reshape(8, -1)[4] += 0.5 * (bx ** 2 + by ** 2 + bz ** 2)
    h = 1.0 / n
    A = U.copy()
    with orc.mhd_reconstruction(recon):
        orc.mhd_run(A, N, N, N, ng, h, h, h, g, [1] * 6, 0.0, 1e300, 3)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Mhd(N, N, N, ng, chl.PREC_FP64_EXACT, reconstruction=RECON[recon])
    hy.run(D, h, h, h, g, 0.0, 1e300, 3)
    assert np.isfinite(A).all()
    real = np.s_[:, ng:N - ng, ng:N - ng, ng:N - ng]
    assert np.array_equal(D.download().reshape(8, N, N, N)[real], A.reshape(8, N, N, N)[real])


@pytest.mark.parametrize("vz", [1e-150, 1e-300, 1e-309, 1e-315])
def test_fp64_form_keeps_tails_bounded(vz):
    """A transverse velocity down to subnormals in a uniform flow is advected: no cell leaves the
    range it started in, by more than the rounding of a subnormal."""
    n, ng, g = 16, 4, 5 / 3
    N = n + 2 * ng
    one = np.ones((N, N, N))
    w = vz * np.random.default_rng(5).uniform(0.5, 1, (N, N, N))
    U = np.stack([one, 0.5 * one, -0.3 * one, w, one / (g - 1) + 0.5 * 0.34 * one]).reshape(-1).copy()
    orc.set_boundaries(U, N, N, N, 5, ng, [1] * 6)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(N, N, N, ng, chl.RECON_PPMC, chl.PREC_FP64)
    hy.run(D, 1 / n, 1 / n, 1 / n, g, 0.0, 1e300, 3)
    out = D.download().reshape(5, -1)
    assert np.isfinite(out).all()
    slack = 1e-12 * vz + 20 * 5e-324
    assert out[3].min() >= 0.5 * vz - slack and out[3].max() <= vz + slack


@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("d_scale,p_scale", [(2.0 ** 60, 2.0 ** 50), (2.0 ** -55, 2.0 ** -55), (2.0 ** -40, 2.0 ** 30)])
def test_mixed_form_far_from_one(recon, d_scale, p_scale):
    """The FP32 quotients where products of two slopes are far from 1 (1e-35 to 1e35, normal in FP32):
    the mixed form's bar on every field that moves."""
    n, ng, g = 16, 4, 5 / 3
    U, N = scaled_box(n, ng, d_scale, p_scale, 0.0)
    h = 1.0 / n
    A = U.copy()
    orc.run(A, N, N, N, ng, 5, h, h, h, g, recon, [1] * 6, 0.0, 1e300, 3)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(N, N, N, ng, RECON[recon], chl.PREC_MIXED)
    hy.run(D, h, h, h, g, 0.0, 1e300, 3)
    a, b = (interior(q, 5, N, N, N, ng) for q in (A, D.download()))
    check_mixed([rel_l1(b[f], a[f]) for f in (0, 1, 2, 4)], names=["density", "momentum_x", "momentum_y", "Energy"])
