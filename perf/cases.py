"""Performance cases of the framework: the steps, stages and snapshot transposes a simulation runs.

Every case is a dict of plain values.  prepare() builds what a simulation has in hand (the
conserved state on the GPU, in torch tensors whose device pointers the library borrows, and the
integrator handle); run() is one pass through the public entry points, advancing the state in
place as a simulation does; work() is the traffic and arithmetic the pass cannot do without;
exact() is the same pass in plain FP64 torch.
"""
import ctypes
import math

import numpy as np
import torch

import cholla_amd as chl

INF = float("inf")
TINY = 1.0e-20
PREC = {"exact": chl.PREC_FP64_EXACT, "fp64": chl.PREC_FP64, "mixed": chl.PREC_MIXED}
RECON = {"plmc": chl.RECON_PLMC, "ppmc": chl.RECON_PPMC}
GHOSTS = {"plmc": 3, "ppmc": 4}
# Floating-point operations of one cell-update, counted from the scheme: each reconstruction and
# Riemann solve once per cell and direction, and the two updates.
FLOPS = {"plmc": 900.0, "ppmc": 1600.0, "mhd": 3000.0}


def listed():
    return [
        # The 1D Sod shock tube at the size the reference's tests and tutorials run: the smallest
        # call there is, a chain of short launches.
        {"name": "sod-1d", "kind": "hydro", "ic": "sod", "nx": 100, "ny": 1, "nz": 1, "recon": "plmc",
         "form": "exact", "steps": 32},
        # The linear-wave system test's box: a small 3D run in the parity form.
        {"name": "linear-wave-64x32x32", "kind": "hydro", "ic": "wave", "nx": 64, "ny": 32, "nz": 32,
         "recon": "plmc", "form": "exact", "steps": 16},
        # A 2D Kelvin-Helmholtz box, not square: parameter studies and tutorials run in 2D.
        {"name": "kh-2d-320x192", "kind": "hydro", "ic": "kh", "nx": 320, "ny": 192, "nz": 1, "recon": "ppmc",
         "form": "fp64", "steps": 16},
        # The drop-in path of a host-driven loop: step, temperature floor, dt and boundaries as
        # separate calls on one small box, the way an unmodified driver calls them.
        {"name": "dropin-48", "kind": "dropin", "ic": "kh", "nx": 48, "ny": 48, "nz": 48, "recon": "plmc",
         "form": "exact", "steps": 4},
        # Cold supersonic gas with dual energy between periodic, reflecting and outflow faces on a
        # ragged box: a wind-and-cloud run, one host-timed grid update per step.
        {"name": "wind-de-120x88x72", "kind": "update", "ic": "wind", "nx": 120, "ny": 88, "nz": 72, "recon": "plmc",
         "form": "fp64", "steps": 4},
        # The Kelvin-Helmholtz box at 256^3 in the parity form: the validation run.
        {"name": "kh-256-exact", "kind": "hydro", "ic": "kh", "nx": 256, "ny": 256, "nz": 256, "recon": "ppmc",
         "form": "exact", "steps": 4},
        # A production FP64 box with sides that no tile divides.
        {"name": "kh-300x212x190-fp64", "kind": "hydro", "ic": "kh", "nx": 300, "ny": 212, "nz": 190, "recon": "ppmc",
         "form": "fp64", "steps": 4},
        # The Kelvin-Helmholtz box at 512^3 in the mixed form: the headline run and the largest.
        {"name": "kh-512-mixed", "kind": "hydro", "ic": "kh", "nx": 512, "ny": 512, "nz": 512, "recon": "ppmc",
         "form": "mixed", "steps": 4},
        # An ensemble of turbulence boxes of uneven sizes, advanced together.
        {"name": "ensemble-64", "kind": "ensemble", "boxes": 64, "recon": "ppmc", "form": "mixed", "steps": 4},
        # Ideal MHD, the Orszag-Tang vortex at 256^3 in the mixed form.
        {"name": "ot-256-mixed", "kind": "mhd", "nx": 256, "ny": 256, "nz": 256, "form": "mixed", "steps": 4},
        # Ideal MHD on a small ragged box in the parity form: test and convergence runs.
        {"name": "ot-56x40x36-exact", "kind": "mhd", "nx": 56, "ny": 40, "nz": 36, "form": "exact", "steps": 8},
        # The snapshot transposes of a whole state: five fields written out and read back.
        {"name": "snapshot-256", "kind": "snapshot", "nx": 256, "ny": 256, "nz": 256, "f32": False},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind by how often it is run, its sizes log-uniform over the range."""
    kind = rng.choice(["1d", "2d", "dropin", "update", "small", "box", "box", "large", "ensemble", "mhd", "mhd", "snapshot"])
    recon = rng.choice(["plmc", "ppmc"])
    if kind == "1d":
        return {"kind": "hydro", "ic": "sod", "nx": _size(rng, 48, 4000), "ny": 1, "nz": 1, "recon": recon,
                "form": rng.choice(["exact", "fp64"]), "steps": 32}
    if kind == "2d":
        return {"kind": "hydro", "ic": "kh", "nx": _size(rng, 64, 900), "ny": _size(rng, 64, 900), "nz": 1,
                "recon": recon, "form": rng.choice(["exact", "fp64"]), "steps": 16}
    if kind == "dropin":
        return {"kind": "dropin", "ic": "kh", "nx": _size(rng, 24, 160), "ny": _size(rng, 24, 160),
                "nz": _size(rng, 24, 160), "recon": recon, "form": "exact", "steps": 4}
    if kind == "update":
        return {"kind": "update", "ic": "wind", "nx": _size(rng, 48, 200), "ny": _size(rng, 48, 200),
                "nz": _size(rng, 48, 200), "recon": recon, "form": rng.choice(["exact", "fp64"]), "steps": 4}
    if kind == "small":
        return {"kind": "hydro", "ic": "wave", "nx": _size(rng, 32, 96), "ny": _size(rng, 16, 64),
                "nz": _size(rng, 16, 64), "recon": recon, "form": rng.choice(["exact", "fp64"]), "steps": 16}
    if kind == "box":
        return {"kind": "hydro", "ic": "kh", "nx": _size(rng, 96, 320), "ny": _size(rng, 96, 320),
                "nz": _size(rng, 96, 320), "recon": recon, "form": rng.choice(["exact", "fp64", "mixed"]), "steps": 4}
    if kind == "large":
        return {"kind": "hydro", "ic": "kh", "nx": _size(rng, 320, 500), "ny": _size(rng, 320, 500),
                "nz": _size(rng, 320, 500), "recon": recon, "form": "mixed", "steps": 4}
    if kind == "ensemble":
        return {"kind": "ensemble", "boxes": _size(rng, 4, 100), "recon": "ppmc",
                "form": rng.choice(["mixed", "fp64"]), "steps": 4}
    if kind == "mhd":
        return {"kind": "mhd", "nx": _size(rng, 32, 256), "ny": _size(rng, 32, 256), "nz": _size(rng, 32, 256),
                "form": rng.choice(["exact", "fp64", "mixed"]), "steps": 4}
    return {"kind": "snapshot", "nx": _size(rng, 32, 300), "ny": _size(rng, 32, 300), "nz": _size(rng, 32, 300),
            "f32": rng.random() < 0.5}


# ------------------------------------------------------------------------------------ inputs
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Borrowed:
    """A contiguous torch tensor as the library borrows it: a device pointer and a length."""

    def __init__(self, t):
        self.t, self.n, self.ptr = t, t.numel(), ctypes.c_void_p(t.data_ptr())


def _ghost(case):
    return 4 if case["kind"] in ("mhd", "snapshot") else GHOSTS[case["recon"]]


def _gamma(case):
    return 1.4 if case.get("ic") == "sod" else 5.0 / 3.0


def _flags(case):
    if case.get("ic") == "sod":
        return [3, 3, 1, 1, 1, 1]
    if case.get("ic") == "wind":
        return [1, 1, 2, 2, 3, 3]
    return [1] * 6


def _widths(case):
    # the linear-wave box is twice as long along x as its y and z sides in the reference's test
    if case.get("ic") == "wave":
        return 1.0 / case["nx"], 0.5 / case["ny"], 0.5 / case["nz"]
    return 1.0 / case["nx"], 1.0 / case["ny"], 1.0 / case["nz"]


def _edges(case, seed):
    """Box edges and rms Mach numbers of an ensemble; the edges are the case's, whatever the seed."""
    r = np.random.default_rng(2024 + case["boxes"])
    edges = r.choice([32, 48, 64, 96, 128], size=case["boxes"])
    return [int(e) for e in edges], np.random.default_rng(seed).uniform(0.5, 3.0, case["boxes"])


def _axes(dims, dev):
    nz, ny, nx = dims
    x = (torch.arange(nx, device=dev, dtype=torch.float64) + 0.5) / nx
    y = (torch.arange(ny, device=dev, dtype=torch.float64) + 0.5) / ny
    z = (torch.arange(nz, device=dev, dtype=torch.float64) + 0.5) / nz
    return x.view(1, 1, -1), y.view(1, -1, 1), z.view(-1, 1, 1)


def _cons(d, v, p, gamma):
    d = d.contiguous()
    return torch.stack([d, d * v[0], d * v[1], d * v[2], p / (gamma - 1.0) + 0.5 * d * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)])


def _interior(case, seed):
    """The real cells of a box at the start of the pass (fields, nz, ny, nx)."""
    dev = _device()
    dims = (case["nz"], case["ny"], case["nx"])
    g = torch.Generator(device=dev).manual_seed(int(seed))
    r = np.random.default_rng(int(seed))
    gamma = _gamma(case)
    x, y, z = _axes(dims, dev)
    one = torch.ones(dims, device=dev, dtype=torch.float64)
    ic = case["ic"]
    if ic == "sod":
        x0 = 0.45 + 0.1 * r.random()
        left = (x < x0) & (one > 0)
        d = torch.where(left, one, 0.1 * one)
        return _cons(d, (0 * one, 0 * one, 0 * one), d.clone(), gamma)
    if ic == "wave":  # a smooth sound wave along x with weak shear waves across it
        s = torch.sin(2 * math.pi * (x + r.random())) * one
        t = torch.sin(2 * math.pi * (y + z + r.random())) * one
        a = 1e-3 * (1 + r.random())
        return _cons(1 + a * s, (a * s, 0.5 * a * t + 0 * s, -0.5 * a * t), 0.6 * (1 + gamma * a * s), gamma)
    if ic == "kh":
        inside = ((y - 0.5).abs() < 0.25) & (one > 0)
        d, vx = torch.where(inside, 2 * one, one), torch.where(inside, 0.5 * one, -0.5 * one)
        noise = 2 * torch.rand(dims, generator=g, device=dev, dtype=torch.float64) - 1
        return _cons(d, (vx, 0.01 * torch.sin(4 * math.pi * (x + r.random())) + 1e-4 * noise, 0 * one), 2.5 * one, gamma)
    # a cold wind over a warm cloud: both sides of the dual-energy switch are present
    ph = 2 * math.pi * r.random(4)
    s = torch.sin(2 * math.pi * x + ph[0]) * torch.cos(2 * math.pi * y + ph[1]) * torch.cos(math.pi * z + ph[2])
    warm = torch.exp(-((x - 0.5) ** 2 + (y - 0.5) ** 2 + (z - 0.5) ** 2) / 0.02)
    d = 1 + 0.3 * s + 2 * warm
    v = (3.0 + 0.2 * s, 0.3 * torch.sin(2 * math.pi * y) * one, 0.2 * torch.sin(math.pi * z + ph[3]) * s)
    p = (2e-4 + 0.5 * warm) * (1 + 0.1 * s)
    U = _cons(d, v, p, gamma)
    return torch.cat([U, (p / (gamma - 1.0)).unsqueeze(0)])


def _turbulence(n, mach, seed, gamma):
    """A solenoidal velocity field of the modes 1 <= |k| <= 4, E(k) ~ k^-2, on unit gas."""
    dev = _device()
    r = np.random.default_rng(int(seed))
    c = 2 * math.pi * (torch.arange(n, device=dev, dtype=torch.float64) + 0.5) / n
    ks = [k for k in np.ndindex(5, 9, 9)]
    ks = np.array([(a, b - 4, d - 4) for a, b, d in ks], dtype=float)
    k2 = (ks ** 2).sum(1)
    ks, k2 = ks[(k2 >= 1) & (k2 <= 16)], k2[(k2 >= 1) & (k2 <= 16)]
    amp = r.normal(size=(len(ks), 2, 3)) / k2[:, None, None]
    amp -= ks[:, None, :] * ((amp * ks[:, None, :]).sum(2) / k2[:, None])[:, :, None]
    # sum over modes of Re[(a - i b) e^(i k.x)], one axis at a time
    w = torch.zeros((3, 9, 9, 5), dtype=torch.complex128)
    for (kx, ky, kz), a in zip(ks.astype(int), amp):
        w[:, kz + 4, ky + 4, kx] += torch.tensor(a[0] - 1j * a[1])
    w = w.to(dev)
    f = [torch.exp(1j * torch.arange(lo, 5, device=dev, dtype=torch.float64).view(-1, 1) * c) for lo in (-4, -4, 0)]
    v = torch.tensordot(w, f[2], dims=([3], [0]))                       # 3, kz, ky, x
    v = torch.tensordot(v, f[1], dims=([2], [0]))                       # 3, kz, x, y
    v = torch.tensordot(v, f[0], dims=([1], [0])).real.permute(0, 3, 2, 1).contiguous()  # 3, z, y, x
    v *= mach * math.sqrt(gamma) / (v ** 2).sum(0).mean().sqrt()
    one = torch.ones((n, n, n), device=dev, dtype=torch.float64)
    return _cons(one, (v[0], v[1], v[2]), one, gamma)


def _orszag_tang(case, seed):
    """The Orszag-Tang vortex with a weak divergence-free z perturbation (8 fields, real cells):
    face fields as the curl of an edge potential, periodic."""
    dev = _device()
    gamma = 5.0 / 3.0
    dims = (case["nz"], case["ny"], case["nx"])
    dx, dy, dz = _widths(case)
    r = np.random.default_rng(int(seed))
    x, y, z = _axes(dims, dev)
    xe, ye, ze = x - 0.5 * dx, y - 0.5 * dy, z - 0.5 * dz  # edges and faces below the cell
    one = torch.ones(dims, device=dev, dtype=torch.float64)
    b0 = 1.0 / math.sqrt(4 * math.pi)
    az = b0 / (4 * math.pi) * (torch.cos(4 * math.pi * xe) + 2 * torch.cos(2 * math.pi * ye)) * one

    def pert():
        a, ph = r.uniform(-1, 1, 4), r.uniform(0, 2 * math.pi, 4)
        return sum(a[m] / (m + 1) * torch.cos(2 * math.pi * (m + 1) * ze + ph[m]) for m in range(4)) * 1e-3 / (2 * math.pi) * one

    ax, ay = pert(), pert()
    up = lambda q, a: torch.roll(q, -1, a)  # noqa: E731
    # the face above each cell: B(i+1/2) = curl of A at that face
    bx = up((up(az, 1) - az) / dy - (up(ay, 0) - ay) / dz, 2)
    by = up((up(ax, 0) - ax) / dz - (up(az, 2) - az) / dx, 1)
    bz = up((up(ay, 2) - ay) / dx - (up(ax, 1) - ax) / dy, 0)
    d = 25.0 / (36.0 * math.pi) * one
    v = (-torch.sin(2 * math.pi * y) * one, torch.sin(2 * math.pi * x) * one, 0 * one)
    U = _cons(d, v, 5.0 / (12.0 * math.pi) * one, gamma)
    for q, a in ((bx, 2), (by, 1), (bz, 0)):
        U[4] += 0.5 * (0.5 * (q + torch.roll(q, 1, a))) ** 2
    return torch.cat([U, bx.unsqueeze(0), by.unsqueeze(0), bz.unsqueeze(0)])


def _pad(V, ng, flags, mhd=False):
    """The state with its ghost cells filled from the real cells V (fields, nz, ny, nx)."""
    nf, nz, ny, nx = V.shape
    gh = [ng if n > 1 else 0 for n in (nz, ny, nx)]
    U = torch.zeros((nf, nz + 2 * gh[0], ny + 2 * gh[1], nx + 2 * gh[2]), device=V.device, dtype=V.dtype)
    U[:, gh[0]:gh[0] + nz, gh[1]:gh[1] + ny, gh[2]:gh[2] + nx] = V
    _fill(U, ng, flags, mhd)
    return U


def _box_inputs(case, seed):
    if case["kind"] == "mhd":
        return _pad(_orszag_tang(case, seed), 4, [1] * 6, True)
    if case["kind"] == "snapshot":
        return _pad(_interior({**case, "ic": "kh"}, seed), 4, [1] * 6)
    return _pad(_interior(case, seed), _ghost(case), _flags(case))


def _dt(case):
    """The host-timed step of the update and drop-in loops: a CFL step with room to spare."""
    vmax = 3.6 if case["ic"] == "wind" else 2.8
    return 0.2 * min(w for w, n in zip(_widths(case), (case["nx"], case["ny"], case["nz"])) if n > 1) / vmax


def prepare(case, seed):
    ng = _ghost(case)
    kind = case["kind"]
    if kind == "ensemble":
        edges, mach = _edges(case, seed)
        gamma = _gamma(case)
        boxes = [_pad(_turbulence(e, m, seed * 1000 + b, gamma), ng, [1] * 6)
                 for b, (e, m) in enumerate(zip(edges, mach))]
        arena = torch.cat([b.reshape(-1) for b in boxes])
        views, at = [], 0
        for b in boxes:
            views.append(_Borrowed(arena[at:at + b.numel()]))
            at += b.numel()
        h = chl.Ensemble([(e + 2 * ng,) * 3 for e in edges], ng, RECON[case["recon"]], PREC[case["form"]],
                         positivity_fallback=True)
        torch.cuda.synchronize()
        h.bind(views, [[1.0 / e] * 3 for e in edges])
        h.start(gamma, U_floor=1e-3)
        return {"case": case, "h": h, "U": arena}
    U = _box_inputs(case, seed).contiguous()
    nz, ny, nx = U.shape[1:]
    s = {"case": case, "U": U, "b": _Borrowed(U), "dims": (nx, ny, nz)}
    if kind == "mhd":
        s["h"] = chl.Mhd(nx, ny, nz, ng, PREC[case["form"]])
    elif kind == "snapshot":
        t = torch.float32 if case["f32"] else torch.float64
        s["buf"] = torch.zeros((5, case["nx"], case["ny"], case["nz"]), device=U.device, dtype=t)
        s["back"] = torch.zeros_like(U)
    else:
        s["h"] = chl.Hydro(nx, ny, nz, ng, RECON[case["recon"]], PREC[case["form"]], bc=_flags(case),
                           dual_energy=case["ic"] == "wind")
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ensemble":
        state["h"].advance(case["steps"])
        return state["U"]
    U, (nx, ny, nz), ng = state["b"], state["dims"], _ghost(case)
    dx, dy, dz = _widths(case)
    if kind in ("hydro", "mhd"):
        steps, t = state["h"].run(U, dx, dy, dz, _gamma(case), 0.0, INF, case["steps"])
        return [state["U"], steps, t]
    if kind == "update":
        dti = [state["h"].update_grid(U, dx, dy, dz, _dt(case), _gamma(case), U_floor=1e-5) for _ in range(case["steps"])]
        return [state["U"], dti]
    if kind == "dropin":
        g, flags, dti = _gamma(case), _flags(case), []
        for _ in range(case["steps"]):
            state["h"].vl_step(U, dx, dy, dz, _dt(case), g)
            chl.apply_temperature_floor(U, nx, ny, nz, ng, 1e-5)
            dti.append(chl.calc_dti(U, nx, ny, nz, ng, dx, dy, dz, g))
            chl.set_boundaries(U, nx, ny, nz, ng, flags)
        return [state["U"], dti]
    # snapshot: every field to its dataset, and (double datasets) back into a grid
    L, c = chl.lib(), (nx, ny, nz, ng, case["nx"], case["ny"], case["nz"], -1)
    pack = L.chl_pack_real_cells_f32 if case["f32"] else L.chl_pack_real_cells
    for f in range(5):
        grid, buf = state["U"][f].data_ptr(), state["buf"][f].data_ptr()
        chl.check(pack(grid, buf, *c))
        if not case["f32"]:
            chl.check(L.chl_unpack_real_cells(buf, state["back"][f].data_ptr(), *c))
    return [state["buf"], state["back"]]


def work(case):
    """Each step reads and writes the FP64 state of the real cells once."""
    if case["kind"] == "ensemble":
        cells = sum(e ** 3 for e in _edges(case, 0)[0])
    else:
        cells = case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "snapshot":
        return {"bytes": 5.0 * cells * (12 if case["f32"] else 32), "flops": 0.0}
    fields = 8 if case["kind"] == "mhd" else (6 if case.get("ic") == "wind" else 5)
    dirs = 1 if case.get("ny") == 1 else (2 if case.get("nz") == 1 else 3)
    flops = FLOPS["mhd"] if case["kind"] == "mhd" else FLOPS[case["recon"]] * dirs / 3
    return {"bytes": 16.0 * fields * cells * case["steps"], "flops": flops * cells * case["steps"]}


# ------------------------------------------------------------------------------------ plain FP64
def exact(case, seed):
    """What run() returns, in plain FP64 torch."""
    kind = case["kind"]
    if kind == "snapshot":
        U = _box_inputs(case, seed)
        V = U[:5, 4:-4, 4:-4, 4:-4].permute(0, 3, 2, 1).contiguous()
        if case["f32"]:
            return [V.to(torch.float32), torch.zeros_like(U)]
        back = torch.zeros_like(U)
        back[:, 4:-4, 4:-4, 4:-4] = U[:, 4:-4, 4:-4, 4:-4]
        return [V, back]
    g = _gamma(case)
    if kind == "ensemble":
        out = []
        for b, (e, m) in enumerate(zip(*_edges(case, seed))):
            U = _pad(_turbulence(e, m, seed * 1000 + b, g), 4, [1] * 6)
            for _ in range(case["steps"]):
                _step(U, 4, case["recon"], g, (1.0 / e,) * 3, 0.3 / _dti(U, 4, g, (1.0 / e,) * 3), 1e-3, fallback=True)
                _fill(U, 4, [1] * 6)
            out.append(U.reshape(-1))
        return torch.cat(out)
    U, ng, w = _box_inputs(case, seed), _ghost(case), _widths(case)
    if kind == "mhd":
        t = 0.0
        for _ in range(case["steps"]):
            dt = 0.3 / _dti_mhd(U, ng, g, w)
            _step_mhd(U, ng, g, w, dt)
            _fill(U, ng, [1] * 6, True)
            t += dt
        return [U, None, t]
    if kind == "hydro":
        t = 0.0
        for _ in range(case["steps"]):
            dt = 0.3 / _dti(U, ng, g, w)
            _step(U, ng, case["recon"], g, w, dt, 0.0)
            _fill(U, ng, _flags(case))
            t += dt
        return [U, None, t]
    dti = []
    for _ in range(case["steps"]):
        _step(U, ng, case["recon"], g, w, _dt(case), 1e-5)
        dti.append(_dti(U, ng, g, w))
        _fill(U, ng, _flags(case))
    return [U, dti]


def _fill(U, ng, flags, mhd=False):
    """Ghost cells of every face in place: 1 periodic, 2 reflecting, 3 outflow (a hydro state's
    ghost keeps no inflowing momentum)."""
    shape = U.shape[1:]
    dev = U.device
    idx, sign = [], []
    for a, n in enumerate(shape):  # axis 0 is z
        i = torch.arange(n, device=dev)
        s = torch.ones(n, device=dev, dtype=U.dtype)
        if n > 1:
            lo, hi = flags[2 * (2 - a)], flags[2 * (2 - a) + 1]
            low, high = i < ng, i >= n - ng
            m = torch.where(low, i + n - 2 * ng if lo == 1 else (2 * ng - 1 - i if lo == 2 else 0 * i + ng), i)
            m = torch.where(high, i - n + 2 * ng if hi == 1 else (2 * (n - ng) - 1 - i if hi == 2 else 0 * i + n - ng - 1), m)
            if lo == 2:
                s = torch.where(low, -s, s)
            if hi == 2:
                s = torch.where(high, -s, s)
            i = m
        idx.append(i)
        sign.append(s)
    for a, n in enumerate(shape):  # x first: later axes copy the corners along
        if shape[2 - a] == 1:
            continue
        ax = 2 - a
        for part in (slice(0, ng), slice(shape[ax] - ng, shape[ax])):
            dst = [slice(None)] * 4
            dst[ax + 1] = part
            new = U.index_select(ax + 1, idx[ax][part])
            s = sign[ax][part].view([-1 if q == ax else 1 for q in range(3)])
            new[3 - ax] = new[3 - ax] * s
            U[tuple(dst)] = new
    if mhd:
        return
    for ax in range(3):
        if shape[ax] == 1:
            continue
        own = [slice(None)] * 3  # a face's own slab: z faces whole planes, y real z, x real y and z
        for q in range(ax):
            if shape[q] > 1:
                own[q] = slice(ng, shape[q] - ng)
        for side, part in enumerate((slice(0, ng), slice(shape[ax] - ng, shape[ax]))):
            if flags[2 * (2 - ax) + side] != 3:
                continue
            sl = list(own)
            sl[ax] = part
            sl = tuple(sl)
            m, d = U[3 - ax][sl], U[0][sl]
            inflow = (m > 0) if side == 0 else (m < 0)
            U[4][sl] = torch.where(inflow, U[4][sl] - 0.5 * m * m / d, U[4][sl])
            U[3 - ax][sl] = torch.where(inflow, 0 * m, m)


def _at(q, axis, k):
    """The value at index i + k along axis (ghost-zone ends wrap, and feed no real cell)."""
    return torch.roll(q, -k, axis)


def _real(U, ng):
    return tuple(slice(ng, n - ng) if n > 1 else slice(None) for n in U.shape[-3:])


def _slabs(U, ng):
    """z-slabs of at most 48 planes with their ghost planes, so large boxes fit; (slab, real k)."""
    nz = U.shape[1]
    if nz <= 64:
        yield U, None
        return
    old = U.clone()
    for k in range(ng, nz - ng, 48):
        e = min(k + 48, nz - ng)
        yield old[:, k - ng:e + ng].clone(), slice(k, e)


def _dti(U, ng, g, w):
    best = 0.0
    V = U[(slice(None),) + _real(U, ng)]
    for k in range(0, V.shape[1], 64):
        d, m, E = V[0, k:k + 64], V[1:4, k:k + 64], V[4, k:k + 64]
        v = m / d
        p = (E - 0.5 * d * (v * v).sum(0)) * (g - 1)
        c = torch.sqrt(g * p / d)
        for a in range(3):
            if U.shape[3 - a] > 1:
                best = max(best, float(((v[a].abs() + c) / w[a]).max()))
    return best


def _recover(U, g):
    """Velocities, pressure and (dual energy) specific internal energy of conserved states."""
    d = U[0]
    v = U[1:4] / d
    kin = 0.5 * d * (v * v).sum(0)
    e = U[4] - kin
    if U.shape[0] == 6:
        e = torch.where(e / U[4] > 1e-3, e, U[5])
    return v, torch.clamp(e * (g - 1), min=TINY)


def _ppm(m2, m1, q, p1, p2):
    """The limited parabola through cells i-2..i+2: its values at cell i's upper and lower faces."""
    dl, dr = q - m1, p1 - q
    sm, s0, sp = 0.5 * dl + 0.5 * (m1 - m2), 0.5 * dr + 0.5 * dl, 0.5 * (p2 - p1) + 0.5 * dr
    R = 0.5 * (m1 + q) + (sm - s0) / 6
    L = 0.5 * (q + p1) + (s0 - sp) / 6
    cm, c0, cp = m2 + q - 2 * m1, m1 + p1 - 2 * q, q + p2 - 2 * p1

    def sgn(t):
        return torch.where(t < 0, -torch.ones_like(t), torch.ones_like(t))

    def face(hi, lo, f, a, b):
        c = 3 * (lo + hi - 2 * f)
        same = (sgn(c) == sgn(a)) & (sgn(c) == sgn(b))
        mag = torch.minimum(1.25 * torch.minimum(a.abs(), b.abs()), c.abs())
        lim = torch.where(same, sgn(c) * mag, 0 * mag)
        return torch.where((f - lo) * (hi - f) < 0, 0.5 * (lo + hi) - lim / 6, f)

    R, L = face(q, m1, R, c0, cm), face(p1, q, L, cp, c0)
    cf = 6 * (R + L - 2 * q)
    same = (sgn(cm) == sgn(c0)) & (sgn(cm) == sgn(cp)) & (sgn(cm) == sgn(cf))
    mag = torch.minimum(1.25 * torch.minimum(torch.minimum(cm.abs(), c0.abs()), cp.abs()), cf.abs())
    lim = torch.where(same, sgn(cf) * mag, 0 * mag)
    top = torch.maximum(torch.maximum(torch.maximum(m2.abs(), m1.abs()), torch.maximum(q.abs(), p1.abs())), p2.abs())
    big = cf.abs() > 1e-12 * top
    rho = torch.where(big, lim / torch.where(big, cf, torch.ones_like(cf)), 0 * cf)
    fl, fr = q - R, L - q
    ext = (fl * fr <= 0) | ((p1 - q) * dl <= 0)
    keep = rho > 1 - 1e-12
    Re, Le = torch.where(keep, R, q - rho * fl), torch.where(keep, L, q + rho * fr)
    Rm = torch.where(fl.abs() >= 2 * fr.abs(), q - 2 * fr, R)
    Lm = torch.where(fr.abs() >= 2 * fl.abs(), q + 2 * fl, L)
    return torch.where(ext, Le, Lm), torch.where(ext, Re, Rm)


def _mono(l, r, c, h):
    lim = torch.minimum(2 * torch.minimum(l.abs(), r.abs()), torch.minimum(c.abs(), h.abs()))
    return torch.where(l * r > 0, torch.copysign(lim, c), 0 * lim)


def _harmonic(l, r):
    ok = l * r > 0
    return torch.where(ok, 2 * l * r / torch.where(ok, l + r, torch.ones_like(l)), 0 * l)


def _clip(f, a, b):
    return torch.minimum(torch.maximum(f, torch.minimum(a, b)), torch.maximum(a, b))


def _states(W, axis, recon, g, fallback):
    """Interface values of the primitives W = [d, vn, v1, v2, p(, e)] at each cell's upper (L) and
    lower (R) face along axis: limited in the cell's characteristic variables."""
    d, p = W[0], W[4]
    c = torch.sqrt(g * p / d)
    c2 = c * c

    def chars(q):
        return [-d * q[1] / (2 * c) + q[4] / (2 * c2), q[0] - q[4] / c2, q[2], q[3], d * q[1] / (2 * c) + q[4] / (2 * c2)]

    def prims(a):
        return [a[0] + a[1] + a[4], c / d * (a[4] - a[0]), a[2], a[3], c2 * (a[0] + a[4])]

    if recon == "ppmc":
        st = {k: chars([_at(q, axis, k) for q in W[:5]]) for k in (-2, -1, 0, 1, 2)}
        L, R = [], []
        for f in range(5):
            l, r = _ppm(*(st[k][f] for k in (-2, -1, 0, 1, 2)))
            L.append(l)
            R.append(r)
        L, R = prims(L), prims(R)
        if fallback:
            ok = (L[0] > 0) & (R[0] > 0) & (L[4] > 0) & (R[4] > 0)
            L, R = [torch.where(ok, q, w) for q, w in zip(L, W)], [torch.where(ok, q, w) for q, w in zip(R, W)]
        ge = [_ppm(*(_at(W[5], axis, k) for k in (-2, -1, 0, 1, 2)))] if len(W) == 6 else []
    else:
        lo, hi = [_at(q, axis, -1) for q in W], [_at(q, axis, 1) for q in W]
        dl, dr = [q - a for q, a in zip(W, lo)], [b - q for q, b in zip(W, hi)]
        dc = [0.5 * (b - a) for a, b in zip(lo, hi)]
        dh = [_harmonic(a, b) for a, b in zip(dl, dr)]
        s = prims([_mono(*q) for q in zip(chars(dl), chars(dr), chars(dc), chars(dh))])
        if len(W) == 6:
            s = s + [_mono(dl[5], dr[5], dc[5], dh[5])]
        L = [_clip(q + 0.5 * t, q, b) for q, t, b in zip(W, s, hi)]
        R = [_clip(q - 0.5 * t, q, a) for q, t, a in zip(W, s, lo)]
        ge = [(L[5], R[5])] if len(W) == 6 else []
    for q in (L, R):
        q[0], q[4] = torch.clamp(q[0], min=TINY), torch.clamp(q[4], min=TINY)
    return (L[:5] + [x[0] for x in ge], R[:5] + [x[1] for x in ge])


def _hllc(l, r, g):
    """HLLC fluxes of the sides [d, vn, v1, v2, p, E(, d*e)] (Roe-averaged signal speeds)."""
    dl, dr = l[0], r[0]
    hl, hr = (l[5] + l[4]) / dl, (r[5] + r[4]) / dr
    sl, sr = torch.sqrt(dl), torch.sqrt(dr)
    avg = lambda a, b: (sl * a + sr * b) / (sl + sr)  # noqa: E731
    v = [avg(l[k], r[k]) for k in (1, 2, 3)]
    a = torch.sqrt(torch.clamp((g - 1) * (avg(hl, hr) - 0.5 * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)), min=0))
    Sl = torch.minimum(v[0] - a, l[1] - torch.sqrt(g * l[4] / dl))
    Sr = torch.maximum(v[0] + a, r[1] + torch.sqrt(g * r[4] / dr))
    Sm = (dr * r[1] * (Sr - r[1]) - dl * l[1] * (Sl - l[1]) + l[4] - r[4]) / (dr * (Sr - r[1]) - dl * (Sl - l[1]))
    ps = dl * (l[1] - Sl) * (l[1] - Sm) + l[4]

    def side(q, S):
        U = [q[0], q[0] * q[1], q[0] * q[2], q[0] * q[3], q[5]] + q[6:]
        F = [U[1], U[1] * q[1] + q[4], U[2] * q[1], U[3] * q[1], (q[5] + q[4]) * q[1]] + [x * q[1] for x in q[6:]]
        ds = q[0] * (S - q[1]) / (S - Sm)
        star = [ds, (U[1] * (S - q[1]) + ps - q[4]) / (S - Sm), ds * q[2], ds * q[3],
                (q[5] * (S - q[1]) - q[4] * q[1] + ps * Sm) / (S - Sm)] + [ds * x / q[0] for x in q[6:]]
        return U, F, star

    Ul, Fl, Al = side(l, Sl)
    Ur, Fr, Ar = side(r, Sr)
    am = Sm.abs()
    out = []
    for k in range(len(Ul)):
        f = 0.5 * (Fl[k] + Fr[k] + (Sr - am) * Ar[k] + (Sl + am) * Al[k] - Sl * Ul[k] - Sr * Ur[k])
        out.append(torch.where(Sl > 0, Fl[k], torch.where(Sr < 0, Fr[k], f)))
    return out


_ROT = {2: (1, 2, 3), 1: (2, 3, 1), 0: (3, 1, 2)}  # momentum fields (normal, t1, t2) by array axis


def _faces(L, R, axis, g, de):
    """HLLC flux at each cell's upper face from L (this cell) and R (the next one), in the state's
    field order; with dual energy the face pressure follows the internal-energy switch."""
    R = [_at(q, axis, 1) for q in R]

    def full(q):
        kin = 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2)
        E = q[4] / (g - 1) + kin
        if not de:
            return q[:5] + [E]
        ge = q[0] * q[5]
        e = torch.where((E - kin) / E > 1e-3, E - kin, ge)
        return q[:4] + [torch.clamp(e * (g - 1), min=TINY), E, ge]

    return _field_order(_hllc(full(L), full(R), g), axis)


def _field_order(f, axis):
    o = list(f)
    for slot, q in zip(_ROT[axis], f[1:4]):
        o[slot] = q
    return o


def _step(U, ng, recon, g, w, dt, u_floor, fallback=False):
    """One van Leer step (piecewise-constant predictor, limited corrector) of U's real cells in
    place, with the temperature floor; dual energy when U has six fields."""
    for V, ks in _slabs(U, ng):
        new = _advance(V, ng, recon, g, w, dt, fallback)
        r = _real(V, ng)
        if ks is None:
            U[(slice(None),) + r] = new[(slice(None),) + r]
        else:
            U[(slice(None), ks) + r[1:]] = new[(slice(None),) + r]
    if U.shape[0] == 6:
        _sync_energies(U, ng)
    r = _real(U, ng)
    if u_floor > 0 and U.shape[1] > 1:
        d = U[0][r]
        kin = 0.5 * (U[1][r] ** 2 + U[2][r] ** 2 + U[3][r] ** 2) / d
        U[4][r] = torch.where((U[4][r] - kin) / d < u_floor, kin + d * u_floor, U[4][r])
        if U.shape[0] == 6:
            U[5][r] = torch.where(U[5][r] / d < u_floor, d * u_floor, U[5][r])


def _advance(U, ng, recon, g, w, dt, fallback):
    nf, de = U.shape[0], U.shape[0] == 6
    axes = [a for a in (2, 1, 0) if U.shape[a + 1] > 1]
    v, p = _recover(U, g)
    H = U.clone()
    for a in axes:
        h = 0.5 * dt / w[2 - a]
        n, t1, t2 = _ROT[a]
        q = [U[0], v[n - 1], v[t1 - 1], v[t2 - 1], p, U[4]] + ([U[5]] if de else [])
        f = _field_order(_hllc(q, [_at(x, a, 1) for x in q], g), a)
        for k in range(nf):
            H[k] += h * (_at(f[k], a, -1) - f[k])
    pdv = None
    if de:
        div = sum(dt / w[2 - a] * (_at(v[2 - a], a, -1) - _at(v[2 - a], a, 1)) for a in axes)
        pdv = 0.5 * p * div
        H[5] += 0.5 * pdv
    v, p = _recover(H, g)
    N = U.clone()
    if de:
        N[5] += pdv
    for a in axes:
        h = dt / w[2 - a]
        n, t1, t2 = _ROT[a]
        W = [H[0], v[n - 1], v[t1 - 1], v[t2 - 1], p] + ([H[5] / H[0]] if de else [])
        L, R = _states(W, a, recon, g, fallback)
        f = _faces(L, R, a, g, de)
        for k in range(nf):
            N[k] += h * (_at(f[k], a, -1) - f[k])
    return N


def _sync_energies(U, ng):
    """The dual-energy selection of the real cells (neighbours clamped to them) and E's sync."""
    V = U[(slice(None),) + _real(U, ng)]
    kin = 0.5 * (V[1] ** 2 + V[2] ** 2 + V[3] ** 2) / V[0]
    tot = V[4] - kin
    top = V[4].clone()
    for a in range(3):
        n = V.shape[a + 1]
        i = torch.arange(n, device=U.device)
        for k in (-1, 1):
            top = torch.maximum(top, V[4].index_select(a, (i + k).clamp(0, n - 1)))
    e = torch.clamp(torch.where((tot / V[4] > 1e-3) | (tot / top > 0.035), tot, V[5]), min=TINY)
    V[5] = e
    V[4] = kin + e


# ------------------------------------------------------------------------------------ plain MHD
def _centred(U):
    return torch.stack([0.5 * (U[5 + q] + _at(U[5 + q], 2 - q, -1)) for q in range(3)])


def _recover_mhd(U, g):
    v, b = U[1:4] / U[0], _centred(U)
    p = (g - 1) * (U[4] - 0.5 * U[0] * (v * v).sum(0) - 0.5 * (b * b).sum(0))
    return v, torch.clamp(p, min=TINY), b


def _fast(d, p, bn, b1, b2, g, s=1.0):
    b2t = bn * bn + b1 * b1 + b2 * b2
    a = g * p + b2t
    return torch.sqrt(torch.clamp((a + s * torch.sqrt(torch.clamp(a * a - 4 * g * p * bn * bn, min=0))) / (2 * d), min=0))


def _dti_mhd(U, ng, g, w):
    best = 0.0
    for V, ks in _slabs(U, ng):
        v, p, b = _recover_mhd(V, g)
        c = _fast(V[0], p, b[0], b[1], b[2], g)
        r = _real(V, ng)
        for a in range(3):
            best = max(best, float(((v[a].abs() + c) / w[a])[r].max()))
    return best


def _hlld(l, r, bn, g):
    """HLLD fluxes of the conserved sides [d, mn, m1, m2, E, b1, b2] with normal field bn."""
    def load(q):
        d = q[0]
        vn, v1, v2 = q[1] / d, q[2] / d, q[3] / d
        mag = 0.5 * (bn * bn + q[5] ** 2 + q[6] ** 2)
        p = torch.clamp((g - 1) * (q[4] - 0.5 * d * (vn * vn + v1 * v1 + v2 * v2) - mag), min=TINY)
        return {"d": d, "v": (vn, v1, v2), "E": q[4], "b": (q[5], q[6]), "p": p, "pt": p + mag}

    def flux(s):
        d, (vn, v1, v2), (b1, b2) = s["d"], s["v"], s["b"]
        return [d * vn, d * vn * vn + s["pt"] - bn * bn, d * vn * v1 - bn * b1, d * vn * v2 - bn * b2,
                vn * (s["E"] + s["pt"]) - bn * (vn * bn + v1 * b1 + v2 * b2), b1 * vn - bn * v1, b2 * vn - bn * v2]

    L, R = load(l), load(r)
    cm = torch.maximum(_fast(L["d"], L["p"], bn, *L["b"], g), _fast(R["d"], R["p"], bn, *R["b"], g))
    SL, SR = torch.minimum(L["v"][0], R["v"][0]) - cm, torch.maximum(L["v"][0], R["v"][0]) + cm
    FL, FR = flux(L), flux(R)
    rl, rr = L["d"] * (SL - L["v"][0]), R["d"] * (SR - R["v"][0])
    M = (rr * R["v"][0] - rl * L["v"][0] - R["pt"] + L["pt"]) / (rr - rl)
    pts = (rr * L["pt"] - rl * R["pt"] + rr * rl * (R["v"][0] - L["v"][0])) / (rr - rl)

    def star(s, S):
        d, (vn, v1, v2), (b1, b2) = s["d"], s["v"], s["b"]
        den = d * (S - vn) * (S - M) - bn * bn
        flat = den.abs() < pts * 1e-8
        safe = torch.where(flat, torch.ones_like(den), den)
        cv = torch.where(flat, 0 * den, bn * (M - vn) / safe)
        cb = torch.where(flat, torch.ones_like(den), (d * (S - vn) ** 2 - bn * bn) / safe)
        w1, w2, c1, c2 = v1 - b1 * cv, v2 - b2 * cv, b1 * cb, b2 * cb
        ds = d * (S - vn) / (S - M)
        E = (s["E"] * (S - vn) - s["pt"] * vn + pts * M + bn * (vn * bn + v1 * b1 + v2 * b2 - M * bn - w1 * c1 - w2 * c2)) / (S - M)
        return {"d": ds, "v": (M, w1, w2), "E": E, "b": (c1, c2)}

    def cons(s):
        return [s["d"], s["d"] * s["v"][0], s["d"] * s["v"][1], s["d"] * s["v"][2], s["E"], s["b"][0], s["b"][1]]

    AL, AR = star(L, SL), star(R, SR)
    ql, qr = torch.sqrt(AL["d"]), torch.sqrt(AR["d"])
    SLs, SRs = M - bn.abs() / ql, M + bn.abs() / qr
    sg = torch.copysign(torch.ones_like(bn), bn)
    weak = 0.5 * bn * bn < 1e-8 * pts
    inv = 1 / (ql + qr)
    up = M >= 0
    vv, bb = [], []
    for k in (0, 1):
        va, vb, ba, bb_ = AL["v"][k + 1], AR["v"][k + 1], AL["b"][k], AR["b"][k]
        vv.append(torch.where(weak, torch.where(up, va, vb), inv * (ql * va + qr * vb + sg * (bb_ - ba))))
        bb.append(torch.where(weak, torch.where(up, ba, bb_), inv * (ql * bb_ + qr * ba + sg * ql * qr * (vb - va))))
    vb_ = M * bn + vv[0] * bb[0] + vv[1] * bb[1]

    def double(s, q, sign):
        dot = M * bn + s["v"][1] * s["b"][0] + s["v"][2] * s["b"][1]
        E = torch.where(weak, s["E"], s["E"] + sign * q * sg * (dot - vb_))
        return {"d": s["d"], "v": (M, vv[0], vv[1]), "E": E, "b": (bb[0], bb[1])}

    DL, DR = double(AL, ql, -1.0), double(AR, qr, 1.0)
    cl, cr, al, ar, el, er = cons(L), cons(R), cons(AL), cons(AR), cons(DL), cons(DR)
    out = []
    for k in range(7):
        fl = FL[k] + SL * (al[k] - cl[k])
        fr = FR[k] + SR * (ar[k] - cr[k])
        f = torch.where(M > 0, fl + SLs * (el[k] - al[k]), fr + SRs * (er[k] - ar[k]))
        f = torch.where(SRs <= 0, fr, f)
        f = torch.where(SLs > 0, fl, f)
        f = torch.where(SR < 0, FR[k], f)
        out.append(torch.where(SL > 0, FL[k], f))
    return out


_TRANS = {0: (1, 2), 1: (2, 0), 2: (0, 1)}  # transverse field components (t1, t2) of direction 0..2


def _mhd_sides(d, v, p_or_E, b, direction, conserved, bn, g):
    """Conserved sides for _hlld from densities, velocities, energy (or pressure) and fields."""
    t1, t2 = _TRANS[direction]
    if conserved:
        E = p_or_E
    else:
        E = p_or_E / (g - 1) + 0.5 * d * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) + 0.5 * (bn ** 2 + b[t1] ** 2 + b[t2] ** 2)
    return [d, d * v[direction], d * v[t1], d * v[t2], E, b[t1], b[t2]]


def _mhd_order(f, direction):
    """[d, mn, m1, m2, E, b1, b2] to (d, mx, my, mz, E) and the two transverse field fluxes."""
    t1, t2 = _TRANS[direction]
    o = [f[0], None, None, None, f[4], f[5], f[6]]
    o[1 + direction], o[1 + t1], o[1 + t2] = f[1], f[2], f[3]
    return o


def _mhd_flux1(U, g):
    v, _, b = _recover_mhd(U, g)
    F = []
    for direction in range(3):
        ax = 2 - direction
        q = _mhd_sides(U[0], v, U[4], b, direction, True, None, g)
        F.append(_mhd_order(_hlld(q, [_at(x, ax, 1) for x in q], U[5 + direction], g), direction))
    return F


def _mhd_plm(d, v, p, b, direction, g):
    """PLMC with the MHD eigenvectors: primitives [d, vn, v1, v2, p, b1, b2] at the upper and lower
    faces of every cell along the direction."""
    ax = 2 - direction
    t1, t2 = _TRANS[direction]
    W = [d, v[direction], v[t1], v[t2], p, b[t1], b[t2]]
    bn = b[direction]
    c = torch.sqrt(g * p / d)
    c2 = c * c
    cf, cs = _fast(d, p, bn, b[t1], b[t2], g), _fast(d, p, bn, b[t1], b[t2], g, -1.0)
    den, n2, n1 = cf ** 2 - cs ** 2, cf ** 2 - c2, c2 - cs ** 2
    one = torch.ones_like(d)
    degenerate = (den <= 0) | (n2 <= 0)
    safe = torch.where(degenerate, one, den)
    af = torch.where(degenerate, one, torch.where(n1 <= 0, 0 * one, torch.sqrt(torch.clamp(n1, min=0) / safe)))
    as_ = torch.where(degenerate, 0 * one, torch.where(n1 <= 0, one, torch.sqrt(torch.clamp(n2, min=0) / safe)))
    bt = torch.sqrt(b[t1] ** 2 + b[t2] ** 2)
    none = bt == 0
    h1 = torch.where(none, one, b[t1] / torch.where(none, one, bt))
    h2 = torch.where(none, 0 * one, b[t2] / torch.where(none, one, bt))
    sg = torch.copysign(one, bn)
    nf, sd = 0.5 / c2, torch.sqrt(d)
    qf, qs = sg * af * cf, sg * as_ * cs
    Af, As = af * c * sd, as_ * c * sd
    Bf, Bs = 0.5 * af / (c * sd), 0.5 * as_ / (c * sd)

    def chars(q):
        par_v, par_b = h1 * q[2] + h2 * q[3], h1 * q[5] + h2 * q[6]
        rot_v, rot_b = h1 * q[3] - h2 * q[2], (h1 * q[6] - h2 * q[5]) * sg / sd
        pd = q[4] / d
        return [nf * af * (pd - cf * q[1]) + nf * qs * par_v + Bs * par_b, 0.5 * (rot_b + rot_v),
                nf * as_ * (pd - cs * q[1]) - nf * qf * par_v - Bf * par_b, q[0] - q[4] / c2,
                nf * as_ * (pd + cs * q[1]) + nf * qf * par_v - Bf * par_b, 0.5 * (rot_b - rot_v),
                nf * af * (pd + cf * q[1]) - nf * qs * par_v + Bs * par_b]

    def prims(a):
        f, s = af * (a[0] + a[6]) + as_ * (a[2] + a[4]), qs * (a[0] - a[6]) + qf * (a[4] - a[2])
        t = As * (a[0] + a[6]) - Af * (a[2] + a[4])
        return [d * f + a[3], cf * af * (a[6] - a[0]) + cs * as_ * (a[4] - a[2]), h1 * s + h2 * (a[5] - a[1]),
                h2 * s + h1 * (a[1] - a[5]), d * c2 * f, h1 * t - h2 * sg * sd * (a[5] + a[1]),
                h2 * t + h1 * sg * sd * (a[5] + a[1])]

    lo, hi = [_at(q, ax, -1) for q in W], [_at(q, ax, 1) for q in W]
    dl, dr = [q - a for q, a in zip(W, lo)], [e - q for q, e in zip(W, hi)]
    dc = [0.5 * (e - a) for a, e in zip(lo, hi)]
    dh = [_harmonic(a, e) for a, e in zip(dl, dr)]
    s = prims([_mono(*q) for q in zip(chars(dl), chars(dr), chars(dc), chars(dh))])
    L = [_clip(q + 0.5 * t, q, e) for q, t, e in zip(W, s, hi)]
    R = [_clip(q - 0.5 * t, q, a) for q, t, a in zip(W, s, lo)]
    for q in (L, R):
        q[0], q[4] = torch.clamp(q[0], min=TINY), torch.clamp(q[4], min=TINY)
    return L, R


def _mhd_flux2(H, g):
    v, p, b = _recover_mhd(H, g)
    F = []
    for direction in range(3):
        ax = 2 - direction
        L, R = _mhd_plm(H[0], v, p, b, direction, g)
        R = [_at(q, ax, 1) for q in R]
        bn = H[5 + direction]

        def side(q):
            E = q[4] / (g - 1) + 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2) + 0.5 * (bn ** 2 + q[5] ** 2 + q[6] ** 2)
            return [q[0], q[0] * q[1], q[0] * q[2], q[0] * q[3], E, q[5], q[6]]

        F.append(_mhd_order(_hlld(side(L), side(R), bn, g), direction))
    return F


def _mhd_edges(F, U):
    """Edge electric fields (Stone & Gardiner 2009, eqs 22-24) at the lower edges of each cell."""
    b = _centred(U)
    cell = [(U[1 + (q + 2) % 3] * b[(q + 1) % 3] - U[1 + (q + 1) % 3] * b[(q + 2) % 3]) / U[0] for q in range(3)]

    def low(q, *dirs):
        for k in dirs:
            q = _at(q, 2 - k, -1)
        return q

    def pick(s, pos, neg):
        return torch.where(s > 0, pos, torch.where(s < 0, neg, 0.5 * (pos + neg)))

    E = []
    for e in range(3):
        a, c = (e + 1) % 3, (e + 2) % 3  # the edge lies along e, at the lower a and c sides
        # E_e on the a faces is -flux of B_c (its first transverse slot is c), on the c faces +flux of B_a
        fa = -F[a][5]
        fc = F[c][6]
        fa, fc = low(fa, a), low(fc, c)  # at the cell's lower faces
        ma, mc = low(F[a][0], a), low(F[c][0], c)
        cc = cell[e]
        # derivatives toward the edge: along c from the a faces, upwinded by the a face's mass flux
        d_c_hi = pick(ma, low(fc, a) - low(cc, a), fc - cc)
        d_c_lo = pick(low(ma, c), low(fc, a) - low(cc, a, c), fc - low(cc, c))
        d_a_hi = pick(mc, low(fa, c) - low(cc, c), fa - cc)
        d_a_lo = pick(low(mc, a), low(fa, c) - low(cc, a, c), fa - low(cc, a))
        E.append(0.25 * (fa + low(fa, c) + fc + low(fc, a) + d_c_hi + d_c_lo + d_a_hi + d_a_lo))
    return E


def _mhd_update(U, F, E, w, dt):
    N = U.clone()
    for direction in range(3):
        h, ax = dt / w[direction], 2 - direction
        for k in range(5):
            N[k] += h * (_at(F[direction][k], ax, -1) - F[direction][k])
    for q in range(3):
        a, c = (q + 1) % 3, (q + 2) % 3
        up = lambda x, *ds: _at(x, 2 - ds[0], 1) if len(ds) == 1 else up(_at(x, 2 - ds[0], 1), *ds[1:])  # noqa: E731
        N[5 + q] += dt / w[c] * (up(E[a], q, c) - up(E[a], q)) - dt / w[a] * (up(E[c], q, a) - up(E[c], q))
    return N


def _step_mhd(U, ng, g, w, dt):
    for V, ks in _slabs(U, ng):
        F = _mhd_flux1(V, g)
        H = _mhd_update(V, F, _mhd_edges(F, V), w, 0.5 * dt)
        F = _mhd_flux2(H, g)
        N = _mhd_update(V, F, _mhd_edges(F, H), w, dt)
        # a real cell's faces, the face below the first one included along a field's own axis
        for f in range(8):
            r = list(_real(V, ng))
            q = None if ks is None else ks
            if f >= 5:
                r[7 - f] = slice(r[7 - f].start - 1, r[7 - f].stop)
                if f == 7 and ks is not None:
                    q = slice(ks.start - 1, ks.stop)
            U[(f, q if q is not None else r[0]) + tuple(r[1:])] = N[f][tuple(r)]
