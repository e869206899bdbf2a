"""The FP64 quotients and square roots of the reference-order form over the exponent range.

The kernels divide without the compiler's range scaling (hydro_physics.hpp: Quot,
SqrtUnscaled), which has IEEE division's bits for numerators of at least 2^-969.  States whose
density, pressure and transverse velocity sit far from 1 (above the scheme's own floors of
1e-20) must therefore stay bit-identical to the CPU oracle."""
import numpy as np
import pytest

import cholla_amd as chl
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


@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("d_scale,p_scale,vz", [(1.0, 1.0, 1e-280), (1.0, 2.0 ** 300, 1e-30),
                                                (2.0 ** 120, 2.0 ** 100, 1e-120), (2.0 ** 200, 2.0 ** -40, 0.0)])
def test_exact_form_bitwise_far_from_one(recon, d_scale, p_scale, vz):
    n, ng, g = 16, 4, 5 / 3
    U, N = scaled_box(n, ng, d_scale, p_scale, vz)
    h = 1.0 / n
    A = U.copy()
    orc.run(A, N, N, N, ng, 5, h, h, h, g, recon, [1] * 6, 0.0, 1e300, 3)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(N, N, N, ng, {orc.PLMC: chl.RECON_PLMC, orc.PPMC: chl.RECON_PPMC}[recon], chl.PREC_FP64_EXACT)
    hy.run(D, h, h, h, g, 0.0, 1e300, 3)
    assert np.isfinite(A).all()
    assert np.array_equal(D.download(), A)
