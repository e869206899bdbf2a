"""The launch shapes the library picks for a box (tile and z planes per workgroup): boxes from
a few cells to several rounds of workgroups, ragged against every tile, bit-identical to the CPU
oracle in the reference-order form and to an explicitly shaped launch in the others."""
import numpy as np
import pytest

import cholla_amd as chl
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
G = 5 / 3


def rough_state(dims, ng, seed, fields=5):
    """A periodic box of smooth waves with noise on every field (dims: real cells x, y, z)."""
    nx, ny, nz = (v + 2 * ng for v in dims)
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(*[(np.arange(n) - ng + 0.5) / r for n, r in ((nz, dims[2]), (ny, dims[1]), (nx, dims[0]))],
                          indexing="ij")
    s = np.sin(2 * np.pi * (x + y)) * np.cos(2 * np.pi * z)
    d = 1 + 0.3 * s + 0.05 * rng.uniform(-1, 1, s.shape)
    v = [0.4 * s, 0.3 * np.cos(2 * np.pi * y) + 0 * s, 0.2 * rng.uniform(-1, 1, s.shape)]
    p = 1 + 0.2 * s
    U = np.stack([d, d * v[0], d * v[1], d * v[2], p / (G - 1) + 0.5 * d * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)])
    U = U.reshape(-1).copy()
    orc.set_boundaries(U, nx, ny, nz, 5, ng, [1] * 6)
    return U, (nx, ny, nz)


# the smallest periodic box of 4 ghost cells, remainders in every axis, one to four planes per workgroup; each is
# under one round of workgroups (test_picked_shape_of_many_rounds has the others)
SIZES = [(4, 5, 4), (33, 17, 5), (24, 24, 24), (70, 9, 50), (130, 66, 36)]


@pytest.mark.parametrize("recon", [orc.PLMC, orc.PPMC])
@pytest.mark.parametrize("dims", SIZES)
def test_picked_shape_matches_oracle(dims, recon):
    ng = 4
    U, (nx, ny, nz) = rough_state(dims, ng, 3)
    w = [1.0 / v for v in dims]
    A = U.copy()
    orc.run(A, nx, ny, nz, ng, 5, *w, G, recon, [1] * 6, 0.0, 1e30, 2)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(nx, ny, nz, ng, {orc.PLMC: chl.RECON_PLMC, orc.PPMC: chl.RECON_PPMC}[recon], chl.PREC_FP64_EXACT)
    hy.run(D, *w, G, 0.0, 1e30, 2)
    assert np.array_equal(D.download(), A), hy.config().kchunk2


@pytest.mark.parametrize("precision", [chl.PREC_FP64, chl.PREC_MIXED])
@pytest.mark.parametrize("dims", SIZES)
def test_picked_shape_matches_explicit(dims, precision):
    ng = 4
    U, (nx, ny, nz) = rough_state(dims, ng, 4)
    w = [1.0 / v for v in dims]
    out = []
    for kw in ({}, dict(tile1=0, tile2=0, kchunk1=32, kchunk2=32)):
        D = chl.DeviceArray.from_host(U)
        hy = chl.Hydro(nx, ny, nz, ng, chl.RECON_PPMC, precision, **kw)
        hy.run(D, *w, G, 0.0, 1e30, 2)
        out.append(D.download())
    # the tiles round alike except where the mixed form's merged lists reorder one sum
    assert np.abs(out[0] - out[1]).max() <= (0 if precision == chl.PREC_FP64 else 4e-16 * np.abs(out[1]).max())


TILES = [(32, 8), (16, 16), (64, 4), (16, 8), (32, 16)]


@pytest.mark.parametrize("precision", [chl.PREC_FP64, chl.PREC_MIXED])
def test_picked_shape_of_many_rounds(precision):
    """A long thin box of more than four rounds of workgroups in both stages, whose picked chunks are
    long: alike with explicit tiles and chunks."""
    ng, dims = 4, (33, 33, 4100)
    U, n = rough_state(dims, ng, 5)
    w = [1.0 / v for v in dims]
    out = []
    for kw in ({}, dict(tile1=0, tile2=0, kchunk1=32, kchunk2=32)):
        D = chl.DeviceArray.from_host(U)
        hy = chl.Hydro(*n, ng, chl.RECON_PPMC, precision, **kw)
        if not kw:
            c = hy.config()
            waves = {1: 4, 2: 3 if precision == chl.PREC_MIXED else 2}  # per SIMD of 256 CUs
            for stage, tile, k, ext in ((1, c.tile1, c.kchunk1, [v + 6 for v in dims]), (2, c.tile2, c.kchunk2, dims)):
                tx, ty = TILES[tile]
                groups = -(-ext[0] // tx) * -(-ext[1] // ty) * -(-ext[2] // k)
                assert k >= 8 and groups > 4 * 256 * waves[stage] * 256 // (tx * ty), (stage, tile, k, groups)
        hy.run(D, *w, G, 0.0, 1e30, 1)
        out.append(D.download())
    assert np.abs(out[0] - out[1]).max() <= (0 if precision == chl.PREC_FP64 else 4e-16 * np.abs(out[1]).max())


def test_picked_ensemble_shape_matches_single_boxes():
    ng, dims = 4, [(8, 8, 8), (20, 12, 40), (33, 33, 33)]
    states, ref = [], []
    for b, d in enumerate(dims):
        U, n = rough_state(d, ng, 7 + b)
        A = U.copy()
        orc.run(A, *n, ng, 5, *[1.0 / v for v in d], G, orc.PPMC, [1] * 6, 0.0, 1e30, 2)
        states.append(chl.DeviceArray.from_host(U))
        ref.append((A, n))
    ens = chl.Ensemble([n for _, n in ref], ng, chl.RECON_PPMC, chl.PREC_FP64_EXACT)
    ens.bind(states, [[1.0 / v for v in d] for d in dims])
    ens.start(G)
    ens.advance(2)
    for D, (A, _) in zip(states, ref):
        assert np.array_equal(D.download(), A)


@pytest.mark.parametrize("recon,ng", [(orc.MHD_PLMC, 4), (orc.MHD_PPMC, 5)])
@pytest.mark.parametrize("dims", [(5, 6, 5), (60, 9, 7), (35, 34, 70), (33, 9, 8300)])
def test_mhd_chunks_match_oracle(dims, recon, ng):
    # a chunk of one plane, remainders along each march, most of a round, more than four rounds at
    # the longest chunks (4 columns of tiles x 519 chunks of 16 planes over 512 slots)
    if recon == orc.MHD_PPMC and dims[2] > 1000:
        pytest.skip("the chunk rule does not depend on the reconstruction")
    U0 = chl.ic_orszag_tang(8, ng, G, seed=5)
    nx, ny, nz = (v + 2 * ng for v in dims)
    V = U0.reshape(8, *(8 + 2 * ng,) * 3)[:, ng:-ng, ng:-ng, ng:-ng]
    ix = [np.arange(-ng, v + ng) % v % 8 for v in (dims[2], dims[1], dims[0])]
    U = V[:, ix[0]][:, :, ix[1]][:, :, :, ix[2]].copy()
    # uniform fields keep div B zero on a box the pattern does not divide
    for f in (5, 6, 7):
        U[4] -= 0.5 * U[f] ** 2
        U[f] = 0.1 * (f - 4)
        U[4] += 0.5 * U[f] ** 2
    U = np.ascontiguousarray(U).reshape(-1)
    w = [1.0 / v for v in dims]
    A = U.copy()
    with orc.mhd_reconstruction(recon):
        orc.mhd_run(A, nx, ny, nz, ng, *w, G, [1] * 6, 0.0, 1e30, 2)
    D = chl.DeviceArray.from_host(U)
    h = chl.Mhd(nx, ny, nz, ng, chl.PREC_FP64_EXACT,
                reconstruction={orc.MHD_PLMC: chl.RECON_PLMC, orc.MHD_PPMC: chl.RECON_PPMC}[recon])
    h.run(D, *w, G, 0.0, 1e30, 2)
    assert np.isfinite(A).all() and np.array_equal(D.download(), A)


@pytest.mark.parametrize("dims", [(4, 4, 4), (4, 5, 4), (65, 5, 9), (63, 33, 17), (96, 40, 44)])
def test_de_sync_columns_match_oracle(dims):
    # columns of 64 x 4: one workgroup, then remainders in x and y, and 4 to 10 planes each
    ng = 4
    U5, (nx, ny, nz) = rough_state(dims, ng, 11)
    U = np.concatenate([U5, np.zeros(nx * ny * nz)])
    a = U.reshape(6, -1)
    a[5] = a[4] - 0.5 * (a[1] ** 2 + a[2] ** 2 + a[3] ** 2) / a[0]
    a[1] += 100.0 * a[0] * (np.arange(a[0].size) // nx % ny < ny // 2)  # a hypersonic slab: both sides of the switch
    a[4] = a[5] + 0.5 * (a[1] ** 2 + a[2] ** 2 + a[3] ** 2) / a[0]
    orc.set_boundaries(U, nx, ny, nz, 6, ng, [1] * 6)
    w = [1.0 / v for v in dims]
    A = U.copy()
    _, t = orc.run(A, nx, ny, nz, ng, 6, *w, G, orc.PLMC, [1] * 6, 0.0, 1e30, 2, dual_energy_on=True)
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(nx, ny, nz, ng, chl.RECON_PLMC, chl.PREC_FP64_EXACT, dual_energy=True)
    _, tg = hy.run(D, *w, G, 0.0, 1e30, 2)
    assert np.isfinite(A).all() and tg == t and np.array_equal(D.download(), A)


@pytest.mark.parametrize("dims,wide", [((122, 40, 20), True), ((250, 34, 9), True), ((130, 66, 36), False)])
def test_mixed_stage1_wide_tiles(dims, wide):
    ng = 4
    U, (nx, ny, nz) = rough_state(dims, ng, 6)
    w = [1.0 / v for v in dims]
    out = []
    for kw in ({}, dict(tile1=0, kchunk1=32)):
        D = chl.DeviceArray.from_host(U)
        hy = chl.Hydro(nx, ny, nz, ng, chl.RECON_PPMC, chl.PREC_MIXED, **kw)
        assert kw or (hy.config().tile1 == 2) == wide
        hy.run(D, *w, G, 0.0, 1e30, 2)
        out.append(D.download())
    assert np.array_equal(out[0], out[1])


def test_autotune_keeps_a_faster_picked_shape():
    """The shapes in hand are among the autotuner's candidates: on a 32^3 box the picked z-chunks
    of one plane run 3-4 times faster than its own list's 8 to 128, and an ensemble's likewise
    (a quarter more).  The bar is half the former factor, for the noise of single launches."""
    ng, dims = 4, (32, 32, 32)
    U, n = rough_state(dims, ng, 8)
    w = [1.0 / v for v in dims]
    D = chl.DeviceArray.from_host(U)
    hy = chl.Hydro(*n, ng, chl.RECON_PLMC, chl.PREC_FP64_EXACT)
    hy.kernel_times(D, *w, G, 2)
    picked = min(sum(hy.kernel_times(D, *w, G, 5)[:2]) for _ in range(4))
    hy.autotune(D, *w, G)
    tuned = min(sum(hy.kernel_times(D, *w, G, 5)[:2]) for _ in range(4))
    assert tuned <= 1.75 * picked, (tuned, picked)
    ens = chl.Ensemble([n] * 2, ng, chl.RECON_PPMC, chl.PREC_MIXED)
    states = [chl.DeviceArray.from_host(U) for _ in range(2)]
    ens.bind(states, [w] * 2)
    ens.start(G)
    chunks = ens.config().kchunk1, ens.config().kchunk2
    cfg = ens.autotune(4)
    assert max(chunks) < 8 and (cfg.launch == chl.LAUNCH_PERSISTENT or min(cfg.kchunk1, cfg.kchunk2) < 8)


@pytest.mark.parametrize("dims,tile", [((8, 8, 8), 1), ((32, 32, 32), 1), ((64, 32, 32), 1), ((40, 40, 40), 4),
                                       ((128, 128, 128), 4)])
def test_plmc_takes_wide_tiles_only_where_narrow_ones_share_a_cu(dims, tile):
    """Stage 2 in FP64 with PLMC: 16x16 tiles while their workgroups are at most one per CU (256),
    where they measure 10-15 % shorter than 32x16."""
    for precision in (chl.PREC_FP64_EXACT, chl.PREC_FP64):
        c = chl.Hydro(*(v + 6 for v in dims), 3, chl.RECON_PLMC, precision).config()
        assert c.tile2 == tile
        assert tile == 4 or np.prod([-(-v // 16) for v in dims[:2]]) * -(-dims[2] // c.kchunk2) <= 256
