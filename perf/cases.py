"""The work a user of this framework has it do, as cases that can be timed.

A simulator's Newton loop calls, per iteration: the flash with its
derivatives, kr/Pc and rock, the residual and the Jacobian, the linear solve
and the update; around it, the save and restore of the last time step.
History matching adds J^T lambda and the parameter gradients; ensembles run
several models at once; a serving loop flashes batches of cells alone.  Each
kind below is one of those calls, through `fim.IsoTFIM`,
`fim.MultiModelBatch` or the C ABI, over the sizes of the repository's own
workloads (1,000-cell grids to a million cells, Nc 2 to 12).

Every context of one model is bound to one stream of the process, as one
simulation's calls follow each other.  Everything is FP64, the only type the framework has.
Flash mappings are the defaults: the autotuner chooses by timing, and another
mapping rounds differently.
"""
import ctypes as C
import math

import numpy as np
import torch

from opencaeporox_amd import abi
from opencaeporox_amd import wells as WL
from opencaeporox_amd import workload as W
from opencaeporox_amd.fim import BATCHED, IsoTFIM, MultiModelBatch

TK = 344.0          # reservoir temperature, K
DT = 1.0            # days
# the solve cases: the small first step after a well event, solved until the solution and not the point
# where the iteration stopped decides the update (as gradient checks and reference runs do)
DT_SOLVE, RTOL, ITS = 0.01, 1e-11, 45

# Fluids of the drawn cases: the 100x100x50 grid's and two more.  Many seeded fluids have a rare composition on which the
# reference's split restarts without end and the framework stops at its cap of 200,000 steps; such a pass takes
# 0.2 to 0.8 s for that one cell.
FLUIDS = (103, 107, 127)

# what the flash leaves behind and the assembly reads (BulkVarSet fields)
FLASH_OUT = ["PHASEEXIST", "S", "XIJ", "RHO", "XI", "MU", "RHOP", "XIP", "MUP", "RHOX", "XIX", "MUX", "NT", "VF",
             "VFP", "VFI", "DSEC_DPRI", "FTYPE_OUT", "SKIP_FLAG", "SKIP_MINEIG", "SKIP_ZI"]
KRPC_OUT = ["KR", "PC", "PJ", "DKRDS", "DPCDS", "PORO", "POROP", "ROCKVP"]


def listed():
    return [
        # one Newton pass of a small model of one reservoir fluid (the 10x10x10 parity grid), replayed from its
        # graph after a restore of the last time step: launches and latency
        {"name": "newton_small", "kind": "newton", "nx": 10, "ny": 10, "nz": 10, "Nc": 6, "fluid": 101, "alpha": 1.0,
         "uniform": True, "graph": True},
        # one Newton pass of an odd-sized sector model, a composition of its own in every cell
        {"name": "newton_sector", "kind": "newton", "nx": 47, "ny": 31, "nz": 23, "Nc": 5, "fluid": 105, "alpha": 1.0,
         "uniform": False, "graph": False},
        # one Newton pass of the 100x100x50 heterogeneous grid, a composition of its own in every cell
        {"name": "newton_field", "kind": "newton", "nx": 100, "ny": 100, "nz": 50, "Nc": 6, "fluid": 103,
         "alpha": 1.0, "uniform": False, "graph": False},
        # the headline workload: a million independent cells of nine components, 30% of them near saturation
        {"name": "flash_million", "kind": "flash", "n": 1048576, "Nc": 9, "fluid": 1102, "alpha": 0.5, "near": 0.3},
        # the flash of a mid-sized model of few components
        {"name": "flash_nc4", "kind": "flash", "n": 150000, "Nc": 4, "fluid": 104, "alpha": 1.0, "near": 0.1},
        # phase equilibrium alone on a caller's device arrays, as a serving loop does it
        {"name": "pe_noalloc", "kind": "pe", "n": 20011, "Nc": 7, "fluid": 107, "alpha": 1.0},
        # kr/Pc, residual and Jacobian from a flash state the caller uploaded, both block sizes of the
        # benchmark: the 100x100x50 grid at b = 8, and an odd grid at b = 7
        {"name": "assemble_b8", "kind": "assemble", "nx": 100, "ny": 100, "nz": 50, "Nc": 6, "fluid": 103},
        {"name": "assemble_b7", "kind": "assemble", "nx": 61, "ny": 45, "nz": 37, "Nc": 5, "fluid": 103},
        # the rest of a Newton iteration after the flash: assembly, device solve and update on the
        # 100x100x50 grid
        {"name": "solve_field", "kind": "solve", "nx": 100, "ny": 100, "nz": 50, "Nc": 6, "fluid": 103,
         "wells": False},
        # the same on a small grid with its five wells' rows in the system
        {"name": "solve_wells", "kind": "solve", "nx": 20, "ny": 20, "nz": 10, "Nc": 6, "fluid": 103, "wells": True},
        # gradients for history matching on the 60x220x85 grid: J^T lambda and dR/d(trans, Vp)
        {"name": "adjoint", "kind": "adjoint", "nx": 60, "ny": 220, "nz": 85, "Nc": 4, "fluid": 104},
        # an ensemble of uneven models, one graph launch for the Newton pass of all of them
        {"name": "ensemble", "kind": "ensemble", "models": 12, "cmin": 3000, "cmax": 20000, "shape": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    """Odd grid of about lo..hi cells, log-uniform, of uneven sides."""
    n = _log_int(rng, lo, hi)
    nz = max(3, min(60, _log_int(rng, 4, 60)))
    ratio = rng.uniform(0.4, 2.5)
    nx = max(3, int(math.sqrt(n / nz * ratio)))
    ny = max(3, int(n / (nx * nz)))
    while nx * ny * nz > hi:
        ny -= 1
    return nx, ny, nz


def draw(rng):
    kind = rng.choice(["newton", "newton", "flash", "flash", "pe", "assemble", "assemble", "solve", "solve", "adjoint",
                       "ensemble"])
    fluid = rng.choice(FLUIDS)
    if kind == "newton":
        nx, ny, nz = _box(rng, 1000, 300000)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "Nc": rng.randint(3, 9), "fluid": fluid, "alpha": 1.0,
                "uniform": rng.random() < 0.5, "graph": rng.random() < 0.5}
    if kind == "flash":
        return {"kind": kind, "n": _log_int(rng, 2000, 400000), "Nc": rng.randint(3, 12), "fluid": fluid,
                "alpha": 0.5 if fluid == 107 else 1.0, "near": rng.choice([0.0, 0.1, 0.3])}
    if kind == "pe":
        return {"kind": kind, "n": _log_int(rng, 2000, 100000), "Nc": rng.randint(2, 9), "fluid": fluid, "alpha": 1.0}
    if kind == "assemble":
        nx, ny, nz = _box(rng, 2000, 500000)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "Nc": rng.randint(3, 9), "fluid": fluid}
    if kind == "solve":
        nx, ny, nz = _box(rng, 2000, 400000)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "Nc": rng.randint(3, 7), "fluid": 103,
                "wells": rng.random() < 0.5}
    if kind == "adjoint":
        nx, ny, nz = _box(rng, 20000, 1000000)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "Nc": rng.randint(3, 6), "fluid": fluid}
    return {"kind": kind, "models": rng.randint(3, 12), "cmin": 2000, "cmax": rng.randint(8000, 30000),
            "shape": rng.randint(10, 1000)}


# ------------------------------------------------------------------ helpers
_stream = None


def _st():
    """The simulation's stream, made at the first use by the HIP runtime the library is linked to (an ordinary
    stream, ordered with the default one, as a C++ program makes it)."""
    global _stream
    if _stream is None:
        _stream = C.c_void_p()
        torch.cuda.init()
        assert abi.load().hipStreamCreate(C.byref(_stream)) == 0
    return _stream


class _Ptr:
    """A device array of a context as torch sees it; holds the context."""

    def __init__(self, owner, ptr, n, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": kind, "data": (ptr, False), "version": 3,
                                         "strides": None}


def _view(dev, ptr, n, kind="<f8"):
    return torch.as_tensor(_Ptr(dev, ptr, n, kind), device="cuda")


def _fields(dev, names):
    out = {}
    for name in names:
        p = C.c_void_p()
        assert dev.lib.ocpx_field_device_ptr(dev.h, abi.FIELD_ID[name], C.byref(p)) == 0
        out[name] = _view(dev, p.value, dev.nb * abi.field_len(name, dev.Nc), "<i4" if name in abi.INT_FIELDS else "<f8")
    return out


def _system(dev):
    """Values and right-hand side of the device block-CSR."""
    p = [C.c_void_p() for _ in range(4)]
    assert dev.lib.ocpx_bsr_device_ptrs(dev.h, *[C.byref(q) for q in p]) == 0
    nnzb = dev.nb + 2 * dev.nconn
    return {"val": _view(dev, p[2].value, nnzb * dev.bs ** 2), "rhs": _view(dev, p[3].value, dev.nb * dev.bs)}


def _gpu(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


class _Batch(MultiModelBatch):
    def __del__(self):
        self.close()


class _Eos:
    """Peng-Robinson in torch, for inputs only (molar volume, stability)."""

    def __init__(self, fluid):
        f = W.fluid_arrays(fluid)
        self.Tc, self.Pc, self.w = _gpu(f["Tc"]), _gpu(f["Pc"]), _gpu(f["acf"])
        self.omk = _gpu(1 - f["kij"])
        w = self.w
        self.m = torch.where(w <= 0.49, 0.37464 + 1.54226 * w - 0.26992 * w ** 2,
                             0.379642 + 1.48503 * w - 0.164423 * w ** 2 + 0.016667 * w ** 3)

    def consts(self, P):
        Pr, Tr = P[:, None] / self.Pc, TK / self.Tc
        A = 0.457235529 * Pr / Tr ** 2 * (1 + self.m * (1 - Tr.sqrt())) ** 2
        return A.sqrt(), 0.077796074 * Pr / Tr

    def z_lnphi(self, c, x):
        sA, Bi = c
        w = sA * x
        s = torch.zeros_like(w)
        for k in range(x.shape[1]):
            s = s + self.omk[k] * w[:, k:k + 1]
        s = sA * s
        A, B = (x * s).sum(1), (x * Bi).sum(1)
        d1, d2 = 1 + math.sqrt(2.0), 1 - math.sqrt(2.0)
        a = (d1 + d2 - 1) * B - 1
        b = A + d1 * d2 * B * B - (d1 + d2) * B * (B + 1)
        cc = -(A * B + d1 * d2 * B * B * (B + 1))
        Q, R = (a * a - 3 * b) / 9, (2 * a ** 3 - 9 * a * b + 27 * cc) / 54
        M = R * R - Q ** 3
        th = torch.acos((R / Q.clamp_min(1e-300) ** 1.5).clamp(-1, 1))
        sq = -2 * Q.clamp_min(0).sqrt()
        r = torch.stack([sq * torch.cos((th + k * 2 * math.pi) / 3) - a / 3 for k in (0, 1, -1)])
        lo, hi = r.amin(0), r.amax(0)
        sM = M.clamp_min(0).sqrt()
        cb = lambda t: t.sign() * t.abs() ** (1.0 / 3)
        one = cb(-R + sM) + cb(-R - sM) - a / 3
        lo = torch.where(lo > B, lo, hi)
        dG = (hi - lo) + torch.log((lo - B) / (hi - B)) - A / (B * (d2 - d1)) * torch.log(
            (lo + d1 * B) * (hi + d2 * B) / ((lo + d2 * B) * (hi + d1 * B)))
        Z = torch.where(M > 0, one, torch.where(dG > 0, lo, hi))
        lg = torch.log((Z + d1 * B) / (Z + d2 * B))
        q = Bi / B[:, None]
        ln = q * (Z - 1)[:, None] - torch.log(Z - B)[:, None] - (A / (d1 - d2) / B * lg)[:, None] * (
            2 * s / A[:, None] - q)
        return Z, ln

    def vm(self, P, x):
        return self.z_lnphi(self.consts(P), x)[0] * W.R_GAS * TK / P

    def unstable(self, P, x, its=25):
        """Whether a Wilson-type trial phase of 25 substitutions has a lower tangent plane."""
        c = self.consts(P)
        d = x.log() + self.z_lnphi(c, x)[1]
        lk = torch.log(self.Pc / P[:, None]) + 5.373 * (1 + self.w) * (1 - self.Tc / TK)
        found = torch.zeros_like(P, dtype=torch.bool)
        for sign in (1.0, -1.0):
            Y = x * torch.exp(sign * lk)
            for _ in range(its):
                y = Y / Y.sum(1, keepdim=True)
                Y = torch.exp(d - self.z_lnphi(c, y)[1])
            far = (((Y / Y.sum(1, keepdim=True)) / x).log() ** 2).sum(1) > 1e-4
            found |= (Y.sum(1) > 1 + 1e-6) & far
        return found

    def psat(self, x):
        """Upper two-phase pressure (NaN without one), good to about 1%."""
        grid = torch.linspace(5.0, 600.0, 16, dtype=torch.float64, device="cuda")
        top = torch.full((x.shape[0],), float("nan"), dtype=torch.float64, device="cuda")
        for p in grid:
            top = torch.where(self.unstable(p.expand(x.shape[0]), x), p, top)
        a, b = top.clone(), top + (grid[1] - grid[0])
        for _ in range(7):
            m = 0.5 * (a + b)
            two = self.unstable(torch.nan_to_num(m, nan=100.0), x)
            a, b = torch.where(two, m, a), torch.where(two, b, m)
        return 0.5 * (a + b)


def _dirichlet(rng, alpha, n, Nc):
    """Dirichlet(0.5) or Dirichlet(1) draws."""
    g = rng.standard_normal((n, Nc)) ** 2 if alpha == 0.5 else rng.standard_exponential((n, Nc))
    g = np.maximum(g, 1e-12)
    return g / g.sum(1, keepdims=True)


def _state(fluid, rock, grid, P, z, rng, perturb):
    """The first Newton flash of a time step: water-only previous phases, the pore space filled at P."""
    nb, Nc = grid.nb, fluid.nc
    nc = Nc + 1
    P = np.round(P, 3)
    vm = _Eos(fluid).vm(_gpu(P), _gpu(z)).cpu().numpy()
    dP = P - rock.Pref
    Vp = grid.v * grid.poro * (1 + (rock.cp1 + rock.cp2 / 2 * dP) * dP)
    Bw = fluid.PVTW[1] * (1 - fluid.PVTW[2] * (P - fluid.PVTW[0]))
    Ni = np.concatenate([z * (Vp * 0.8 / vm)[:, None], (Vp * 0.2 / Bw)[:, None]], axis=1)
    lNi = Ni
    if perturb:
        Ni = Ni * (1 + rng.uniform(-0.01, 0.01, Ni.shape))
        P = P + np.round(rng.uniform(-1.0, 1.0, nb), 3)
    x = np.zeros((nb, 3, nc))
    x[:, 2, Nc] = 1.0
    return {"P": P, "T": np.full(nb, TK - W.CONV4), "NI": Ni.ravel(), "LNI": lNi.ravel(),
            "PHASEEXIST": np.tile(np.array([0, 0, 1], np.uint32), nb), "S": np.tile(np.array([0.0, 0.0, 1.0]), nb),
            "XIJ": x.ravel()}


def _reservoir(case, rng):
    """Heterogeneous Cartesian grid, hydrostatic pressures with a spread, one composition or one per cell."""
    nx, ny, nz, Nc = case["nx"], case["ny"], case["nz"], case["Nc"]
    nb = nx * ny * nz
    k = np.exp(rng.normal(np.log(100.0), case.get("sigma", 2.0), nb))
    grid = W.cartesian_grid(nx, ny, nz, 6.096, k, k, 0.1 * k, rng.uniform(0.1, 0.3, nb))
    fluid, rock = W.make_fluid(Nc, case["fluid"]), W.make_rock()
    P = 200.0 + 0.0980665 * (grid.depth - grid.depth.min()) + rng.normal(0, 10.0, nb)
    # one reservoir fluid (the moles then move by up to 1% per cell), or a composition of its own in every cell
    z = _dirichlet(rng, case.get("alpha", 1.0), 1 if case.get("uniform", True) else nb, Nc)
    z = np.broadcast_to(z, (nb, Nc)).copy()
    return W.Workload(case["kind"], fluid, W.make_sat(), rock, grid, _state(fluid, rock, grid, P, z, rng, True))


# ------------------------------------------- a flash state a caller uploads
def _flashed(case, seed):
    """Grid and the state a flash leaves, drawn instead of computed: phases, saturations, compositions, the
    phase properties and their derivatives at the magnitudes of an oil-gas-water reservoir.  Cell-major arrays
    on the GPU."""
    rng = np.random.Generator(np.random.PCG64(seed))
    nx, ny, nz, Nc = case["nx"], case["ny"], case["nz"], case["Nc"]
    nb, nc, B = nx * ny * nz, Nc + 1, Nc + 2
    k = np.exp(rng.normal(np.log(100.0), 2.0, nb))
    grid = W.cartesian_grid(nx, ny, nz, 6.096, k, k, 0.1 * k, rng.uniform(0.1, 0.3, nb))
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 77)
    U = lambda lo, hi, *s: lo + (hi - lo) * torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)
    N = lambda s, *n: s * torch.randn(*n, generator=g, device="cuda", dtype=torch.float64)
    kind = torch.rand(nb, generator=g, device="cuda")
    ex = torch.ones(nb, 3, dtype=torch.bool, device="cuda")
    ex[:, 0] = kind > 0.2                       # a fifth gas-water, two fifths oil-water, the rest three phases
    ex[:, 1] = (kind <= 0.2) | (kind > 0.6)
    S = U(0.05, 1.0, nb, 3) * ex
    S = S / S.sum(1, keepdim=True)
    x = torch.zeros(nb, 3, nc, dtype=torch.float64, device="cuda")
    for j in (0, 1):
        y = -torch.log(U(1e-6, 1.0, nb, Nc))
        x[:, j, :Nc] = y / y.sum(1, keepdim=True) * ex[:, j:j + 1]
    x[:, 2, Nc] = 1.0
    rho = torch.stack([U(550, 850, nb), U(80, 250, nb), U(990, 1020, nb)], 1)
    xi = torch.stack([U(4, 9, nb), U(3, 12, nb), U(0.98, 1.02, nb)], 1)
    mu = torch.stack([U(0.2, 2.0, nb), U(0.01, 0.05, nb), U(0.65, 0.75, nb)], 1)
    hc = torch.tensor([1.0, 1.0, 0.0], dtype=torch.float64, device="cuda")
    vec = lambda v: torch.cat([v[:, :, :Nc] * hc[None, :, None], torch.zeros(nb, 3, 1, dtype=torch.float64, device="cuda")], 2)
    P = torch.round((200 + 0.0980665 * (_gpu(grid.depth) - float(grid.depth.min())) + N(10.0, nb)) * 1000) / 1000
    vf = _gpu(grid.v * grid.poro) * U(0.98, 1.02, nb)
    Nt = vf * U(3.0, 6.0, nb)
    y = -torch.log(U(1e-6, 1.0, nb, nc))
    Ni = Nt[:, None] * y / y.sum(1, keepdim=True)
    X = torch.zeros(nb, 3 + 3 * nc, B, dtype=torch.float64, device="cuda")
    X[:, :3, 0] = N(2e-3, nb, 3)
    X[:, :3, 1:] = N(0.5, nb, 3, nc) / Nt[:, None, None]
    X[:, :3] *= ex[:, :, None]
    for j in (0, 1):
        rows = slice(3 + j * nc, 3 + j * nc + Nc)
        X[:, rows, 0] = N(1e-3, nb, Nc) * ex[:, j:j + 1]
        X[:, rows, 1:1 + Nc] = N(0.5, nb, Nc, Nc) / Nt[:, None, None] * ex[:, j:j + 1, None]
    f = {"P": P, "NI": Ni, "LNI": Ni * U(0.99, 1.01, nb, nc), "PHASEEXIST": ex, "S": S, "XIJ": x, "RHO": rho * ex,
         "XI": xi * ex, "MU": torch.where(ex, mu, 1.0), "RHOP": U(0.02, 0.3, nb, 3) * ex, "XIP": xi * U(1e-4, 3e-3, nb, 3) * ex,
         "MUP": mu * N(2e-3, nb, 3) * ex, "RHOX": vec(N(300.0, nb, 3, nc)) * ex[:, :, None],
         "XIX": vec(N(4.0, nb, 3, nc)) * ex[:, :, None], "MUX": vec(N(1.0, nb, 3, nc) * mu[:, :, None]) * ex[:, :, None],
         "NT": Nt, "VF": vf, "VFP": -vf * U(1e-4, 5e-3, nb), "VFI": U(0.1, 0.4, nb, nc), "DSEC_DPRI": X}
    return grid, f


def _upload(case, seed):
    grid, f = _flashed(case, seed)
    dev = IsoTFIM(W.make_fluid(case["Nc"], case["fluid"]), W.make_sat(), W.make_rock(), grid, _st())
    dev.set("T", np.full(grid.nb, TK - W.CONV4))
    for name, v in f.items():
        dev.set(name, (v.to(torch.int32) if v.dtype == torch.bool else v).cpu().numpy())
    return dev


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    rng = np.random.Generator(np.random.PCG64(int(seed)))
    s = _PREPARE[case["kind"]](case, rng, int(seed))
    torch.cuda.synchronize()
    return s


def _prepare_newton(case, rng, seed):
    dev = IsoTFIM.from_workload(_reservoir(case, rng), _st())
    dev.UpdateLastTimeStep()
    return {"kind": "newton", "dev": dev, "graph": case["graph"],
            "out": {**_system(dev), **_fields(dev, FLASH_OUT + KRPC_OUT)}}


def _prepare_flash(case, rng, seed):
    n, Nc = case["n"], case["Nc"]
    fluid, rock = W.make_fluid(Nc, case["fluid"]), W.make_rock()
    e = np.zeros(0)
    grid = W.Grid(n, 1, 1, np.full(n, 226.5), np.full(n, 2000.0), np.full(n, 0.2), e.astype(np.int32),
                  e.astype(np.int32), e)
    z = _dirichlet(rng, case["alpha"], n, Nc)
    P = rng.uniform(100.0, 280.0, n)
    near = np.where(rng.uniform(0, 1, n) < case["near"])[0]
    if near.size:
        ps = _Eos(fluid).psat(_gpu(z[near])).cpu().numpy()
        P[near] = np.where(np.isfinite(ps), ps * (1 + rng.uniform(-0.05, 0.05, near.size)), P[near])
    wl = W.Workload("flash", fluid, W.make_sat(), rock, grid, _state(fluid, rock, grid, P, z, rng, False))
    dev = IsoTFIM.from_workload(wl, _st())
    dev.UpdateLastTimeStep()
    return {"kind": "flash", "dev": dev, "out": _fields(dev, FLASH_OUT + ["ITERS"])}


def _prepare_pe(case, rng, seed):
    n, Nc = case["n"], case["Nc"]
    z = _dirichlet(rng, case["alpha"], n, Nc)
    d = lambda *s: torch.empty(*s, dtype=torch.float64, device="cuda")
    i = lambda: torch.empty(n, dtype=torch.int32, device="cuda")
    return {"kind": "pe", "fluid": W.make_fluid(Nc, case["fluid"]), "n": n, "lib": abi.load(),
            "P": _gpu(np.round(rng.uniform(20.0, 280.0, n), 3)), "T": _gpu(np.full(n, TK - W.CONV4)),
            "z": _gpu(z.T), "out": {"NP": i(), "nu": d(n), "x": d(2 * Nc, n), "ftype": i()}}


def _prepare_assemble(case, rng, seed):
    dev = _upload(case, seed)
    return {"kind": "assemble", "dev": dev, "out": {**_system(dev), **_fields(dev, KRPC_OUT)}}


def _prepare_solve(case, rng, seed):
    wl = _reservoir({**case, "uniform": True, "sigma": 1.0}, rng)
    dev = IsoTFIM.from_workload(wl, _st())
    dev.newton_pass(DT, BATCHED)
    dev.UpdateLastTimeStep()
    ws = WL.corner_and_centre_wells(wl) if case["wells"] else []
    s = {"kind": "solve", "dev": dev, "bhp": np.array([w.bhp for w in ws])}
    if ws:
        dev.SetWells(ws)
    s["out"] = {**_system(dev), **_fields(dev, ["P", "NI", "S", "XIJ"])}
    run(s)              # a program's context has its solver set up (hierarchy, colouring, Krylov vectors)
    return s


def _prepare_adjoint(case, rng, seed):
    dev = _upload(case, seed)
    dev.CalKrPc()
    dev.AssembleMatBulks(DT)
    d = lambda n: torch.empty(n, dtype=torch.float64, device="cuda")
    return {"kind": "adjoint", "dev": dev, "lam": _lambda(dev.nb * dev.bs, seed),
            "out": {"gX": d(dev.nb * dev.bs), "gT": d(dev.nconn), "gV": d(dev.nb)}}


def _lambda(n, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 13)
    return torch.randn(n, generator=g, dtype=torch.float64, device="cuda")


def _prepare_ensemble(case, rng, seed):
    sizes = np.random.Generator(np.random.PCG64(case["shape"]))      # the ensemble's shape is the case's, not the seed's
    wls = []
    for m in range(case["models"]):
        nx, ny, nz = W.model_box(int(np.exp(sizes.uniform(np.log(case["cmin"]), np.log(case["cmax"])))))
        Nc = int(sizes.integers(3, 13))
        nb = nx * ny * nz
        k = np.exp(rng.normal(np.log(100.0), 1.0, nb))
        grid = W.cartesian_grid(nx, ny, nz, 6.096, k, k, 0.1 * k, rng.uniform(0.1, 0.3, nb))
        fluid, rock = W.make_fluid(Nc, FLUIDS[m % 3]), W.make_rock()
        st = _state(fluid, rock, grid, rng.uniform(100.0, 280.0, nb), _dirichlet(rng, 1.0, nb, Nc), rng, True)
        wls.append(W.Workload(f"model {m}", fluid, W.make_sat(), rock, grid, st))
    batch = _Batch(wls)
    batch.UpdateLastTimeStep()
    outs = {str(Nc): {**_system(d), **_fields(d, ["S", "XIJ", "PHASEEXIST"])} for Nc, (d, _) in batch.groups.items()}
    for g in outs.values():                                          # the views keep the batch
        for t in g.values():
            t._batch = batch
    return {"kind": "ensemble", "batch": batch, "out": outs}


_PREPARE = {"newton": _prepare_newton, "flash": _prepare_flash, "pe": _prepare_pe, "assemble": _prepare_assemble,
            "solve": _prepare_solve, "adjoint": _prepare_adjoint, "ensemble": _prepare_ensemble}


# ---------------------------------------------------------------------- run
def run(s):
    kind = s["kind"]
    if kind == "pe":
        o = s["out"]
        rc = s["lib"].ocpx_phase_equilibrium_noalloc(
            C.byref(s["fluid"]), s["n"], s["P"].data_ptr(), s["T"].data_ptr(), s["z"].data_ptr(), o["NP"].data_ptr(),
            o["nu"].data_ptr(), o["x"].data_ptr(), o["ftype"].data_ptr(), _st())
        assert rc == 0
    elif kind == "ensemble":
        s["batch"].ResetToLastTimeStep()
        s["batch"].newton_pass(DT, graph=True)
        s["batch"].sync()                   # every step of an ensemble ends in a convergence check
    else:
        dev = s["dev"]
        if kind == "newton":
            dev.ResetToLastTimeStep()
            dev.newton_pass(DT, BATCHED, graph=s["graph"])
        elif kind == "flash":
            dev.ResetToLastTimeStep()
            dev.CalFlash(BATCHED)
        elif kind == "assemble":
            dev.CalKrPc()
            dev.AssembleMatBulks(DT)
        elif kind == "solve":
            dev.ResetToLastTimeStep()
            dev.CalKrPc()
            dev.AssembleMatBulks(DT_SOLVE)
            if s["bhp"].size:
                dev.set_well_bhp(s["bhp"])
                dev.CalResWells(DT_SOLVE, jacobian=True)
            _, its, _ = dev.LinearSolve(RTOL, 200, fetch=False)
            if its > 0:                     # else a program cuts the time step
                dev.GetSolution()
        else:
            o = s["out"]
            dev.jt_lambda_dev(s["lam"].data_ptr(), o["gX"].data_ptr())
            dev.dR_dparams_dev(DT, s["lam"].data_ptr(), o["gT"].data_ptr(), o["gV"].data_ptr())
    return s["out"]


# --------------------------------------------------------------------- work
def _conns(nx, ny, nz):
    return (nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1)


def _flash_work(n, Nc):
    """Inputs and outputs of the flash with derivatives once; flops at the 190 fugacity evaluations per cell
    the mixed workload takes on average."""
    nc, b = Nc + 1, Nc + 2
    byts = 8 * n * (2 + nc + 3 + 3 * nc + 8) + 8 * n * (3 * b * b + 9 * nc + 3 * nc + 24 + nc + Nc)
    return byts, 190.0 * n * (2 * Nc * Nc + 16 * Nc + 60)


def _assembly_bytes(n, nconn, Nc):
    """Cell state read once, Jacobian and residual written once."""
    nc, np_, b = Nc + 1, 3, Nc + 2
    return n * (8 * (np_ * (9 + 2 * np_ + 4 * nc) + 3 + nc + np_ * b * b) + 8 * (b * b + b)) + nconn * (24 + 16 * b * b)


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        rng = np.random.Generator(np.random.PCG64(case["shape"]))
        byts = flops = 0.0
        for _ in range(case["models"]):
            box = W.model_box(int(np.exp(rng.uniform(np.log(case["cmin"]), np.log(case["cmax"])))))
            Nc = int(rng.integers(3, 13))
            n = box[0] * box[1] * box[2]
            fb, ff = _flash_work(n, Nc)
            byts += fb + _assembly_bytes(n, _conns(*box), Nc)
            flops += ff
        return {"bytes": byts, "flops": flops}
    Nc = case["Nc"]
    if kind == "flash":
        b, f = _flash_work(case["n"], Nc)
        return {"bytes": b, "flops": f}
    if kind == "pe":
        return {"bytes": 8.0 * case["n"] * (2 + Nc + 1 + 2 * Nc + 1), "flops": _flash_work(case["n"], Nc)[1]}
    box = case["nx"], case["ny"], case["nz"]
    n, c, b = box[0] * box[1] * box[2], _conns(*box), Nc + 2
    if kind == "newton":
        fb, ff = _flash_work(n, Nc)
        return {"bytes": fb + _assembly_bytes(n, c, Nc), "flops": ff + 60.0 * c * b * b}
    if kind == "assemble":
        return {"bytes": _assembly_bytes(n, c, Nc), "flops": 60.0 * c * b * b}
    if kind == "adjoint":
        return {"bytes": 8.0 * ((n + 2 * c) * b * b + 2 * n * b + 2 * c + n + n * 3 * (6 + Nc + 1)),
                "flops": 2.0 * (n + 2 * c) * b * b}
    # assembly, iterations that read the matrix once each, update
    return {"bytes": _assembly_bytes(n, c, Nc) + ITS * 8.0 * (n + 2 * c) * b * b + 8.0 * n * 3 * b * b,
            "flops": ITS * 2.0 * (n + 2 * c) * b * b}


# -------------------------------------------------------------------- exact
def _table(rows, ncol, v):
    t = _gpu(np.array(rows).reshape(-1, ncol))
    i = torch.searchsorted(t[:, 0].contiguous(), v, right=True)
    k = (i - 1).clamp(0, t.shape[0] - 2)
    inside = (i > 0) & (i < t.shape[0])
    sl = torch.where(inside[:, None], (t[k + 1] - t[k]) / (t[k + 1, :1] - t[k, :1]), 0.0)
    end = torch.where(i > 0, t.shape[0] - 1, 0)
    return torch.where(inside[:, None], t[k] + sl * (v - t[k, 0])[:, None], t[end]), sl


def _krpc(f, grid):
    """kr, Pc and their slopes (two-table Stone II), rock."""
    sat, rock = W.make_sat(), W.make_rock()
    S = f["S"]
    nb = S.shape[0]
    w, dw = _table(sat.swof[:4 * sat.nswof], 4, S[:, 2].contiguous())
    g, dg = _table(sat.sgof[:4 * sat.nsgof], 4, S[:, 1].contiguous())
    c = sat.swof[2]
    kr, pc = torch.zeros(nb, 3, dtype=torch.float64, device="cuda"), torch.zeros(nb, 3, dtype=torch.float64, device="cuda")
    dk, dp = torch.zeros(nb, 3, 3, dtype=torch.float64, device="cuda"), torch.zeros(nb, 3, 3, dtype=torch.float64, device="cuda")
    kr[:, 2], kr[:, 1], pc[:, 2], pc[:, 1] = w[:, 1], g[:, 1], -w[:, 3], g[:, 3]
    kr0 = c * ((w[:, 2] / c + w[:, 1]) * (g[:, 2] / c + g[:, 1]) - (w[:, 1] + g[:, 1]))
    ok = kr0 >= 0
    kr[:, 0] = torch.where(ok, kr0, 0.0)
    dk[:, 2, 2], dk[:, 1, 1], dp[:, 2, 2], dp[:, 1, 1] = dw[:, 1], dg[:, 1], -dw[:, 3], dg[:, 3]
    dk[:, 0, 2] = torch.where(ok, c * ((dw[:, 2] / c + dw[:, 1]) * (g[:, 2] / c + g[:, 1]) - dw[:, 1]), 0.0)
    dk[:, 0, 1] = torch.where(ok, c * ((w[:, 2] / c + w[:, 1]) * (dg[:, 2] / c + dg[:, 1]) - dg[:, 1]), 0.0)
    dP = f["P"] - rock.Pref
    poro0 = _gpu(grid.poro)
    poro = poro0 * (1 + (rock.cp1 + rock.cp2 / 2 * dP) * dP)
    return kr, pc, dk, dp, poro, poro0 * (rock.cp1 + rock.cp2 * dP), _gpu(grid.v) * poro


def _fluxes(f, grid, kr, pc, lo, hi):
    """Per connection lo..hi: phase flux factors dPhi, upstream cell, active flag (two-point, upwinded)."""
    b = torch.as_tensor(grid.conn_b[lo:hi], dtype=torch.int64, device="cuda")
    e = torch.as_tensor(grid.conn_e[lo:hi], dtype=torch.int64, device="cuda")
    ex, rho, G, z = f["PHASEEXIST"], f["RHO"], 0.0000980665, _gpu(grid.depth)
    Pj = f["P"][:, None] + pc
    xb, xe = ex[b], ex[e]
    r = torch.where(xb & xe, (rho[b] + rho[e]) / 2, torch.where(xb, rho[b], rho[e]))
    dPhi = (Pj[b] - G * r * z[b][:, None]) - (Pj[e] - G * r * z[e][:, None])
    up = ~(dPhi < 0)
    act = (xb | xe) & torch.where(up, xb, xe)
    both = torch.where(up, xe, xb)                       # the downstream cell has the phase too
    return b, e, dPhi, up, act, both, G * (z[b] - z[e]), Pj


def _exact_assemble(case, seed):
    grid, f = _flashed(case, seed)
    kr, pc, dk, dp, poro, poroP, Vp = _krpc(f, grid)
    nb, nconn, nc = grid.nb, grid.nconn, case["Nc"] + 1
    B = nc + 1
    X, ex = f["DSEC_DPRI"], f["PHASEEXIST"]
    dS, dx = X[:, :3], X[:, 3:].reshape(nb, 3, nc, B)
    one = torch.zeros(B, dtype=torch.float64, device="cuda")
    one[0] = 1.0
    chain = lambda p, v: f[p][:, :, None] * one + (f[v][:, :, None, :] @ dx)[:, :, 0]
    drho, dxi, dmu = chain("RHOP", "RHOX"), chain("XIP", "XIX"), chain("MUP", "MUX")
    dkr, dPj = dk @ dS, one + dp @ dS
    xi, mu = f["XI"], f["MU"]
    lam = torch.where(ex, xi * kr / mu, 0.0)
    q = lambda t: t[:, :, None]
    dlam = torch.where(q(ex), q(kr / mu) * dxi + q(xi / mu) * dkr - q(xi * kr / (mu * mu)) * dmu, 0.0)
    drho = torch.where(q(ex), drho, 0.0)
    # accumulation
    diag = torch.zeros(nb, B, B, dtype=torch.float64, device="cuda")
    diag[:, 0, 0] = _gpu(grid.v) * poroP - f["VFP"]
    diag[:, 0, 1:] = -f["VFI"]
    idx = torch.arange(1, B, device="cuda")
    diag[:, idx, idx] = 1.0
    res = torch.cat([(Vp - f["VF"])[:, None], f["NI"] - f["LNI"]], 1)
    # slots: the diagonal, then the row's connections in connection order
    cb, ce = (torch.as_tensor(a, dtype=torch.int64, device="cuda") for a in (grid.conn_b, grid.conn_e))
    k = torch.arange(nconn, device="cuda")
    row = torch.cat([torch.arange(nb, device="cuda"), cb, ce])
    key = torch.cat([torch.full((nb,), -1, device="cuda"), k, k])
    slot = torch.empty(nb + 2 * nconn, dtype=torch.int64, device="cuda")
    slot[torch.argsort(row * (nconn + 2) + key)] = torch.arange(nb + 2 * nconn, device="cuda")
    val = torch.zeros(nb + 2 * nconn, B, B, dtype=torch.float64, device="cuda")
    T = _gpu(grid.trans)
    step = 200000
    for lo in range(0, nconn, step):
        hi = min(nconn, lo + step)
        b, e, dPhi, up, act, both, dG, _ = _fluxes(f, grid, kr, pc, lo, hi)
        m = hi - lo
        Eb = torch.zeros(m, nc, B, dtype=torch.float64, device="cuda")
        Ee, F = torch.zeros_like(Eb), torch.zeros(m, nc, dtype=torch.float64, device="cuda")
        for j in range(3):
            u = torch.where(up[:, j], b, e)
            a = torch.where(act[:, j], T[lo:hi], 0.0)
            xu, lu = f["XIJ"][u, j], lam[u, j]
            F += (a * lu * dPhi[:, j])[:, None] * xu
            wU, wD = torch.where(both[:, j], 0.5, 1.0), torch.where(both[:, j], 0.5, 0.0)
            wb, we = torch.where(up[:, j], wU, wD), torch.where(up[:, j], wD, wU)
            vb = dPj[b, j] - (dG * wb)[:, None] * drho[b, j]
            ve = -dPj[e, j] - (dG * we)[:, None] * drho[e, j]
            c = (a * lu)[:, None] * xu
            own = (a * dPhi[:, j])[:, None, None] * (xu[:, :, None] * dlam[u, j][:, None, :] + lu[:, None, None] * dx[u, j])
            isb = up[:, j][:, None, None]
            Eb += c[:, :, None] * vb[:, None, :] + torch.where(isb, own, 0.0)
            Ee += c[:, :, None] * ve[:, None, :] + torch.where(isb, 0.0, own)
        sb, se = slot[nb + lo:nb + hi], slot[nb + nconn + lo:nb + nconn + hi]
        val[sb, 1:] = DT * Ee
        val[se, 1:] = -DT * Eb
        diag[:, 1:].index_add_(0, b, DT * Eb)
        diag[:, 1:].index_add_(0, e, -DT * Ee)
        res[:, 1:].index_add_(0, b, DT * F)
        res[:, 1:].index_add_(0, e, -DT * F)
    val[slot[:nb]] = diag
    soa = lambda t: t.reshape(nb, -1).t().contiguous().reshape(-1)
    out = {"val": val.reshape(-1), "rhs": -res.reshape(-1), "KR": soa(kr), "PC": soa(pc), "PJ": soa(f["P"][:, None] + pc),
           "DKRDS": soa(dk), "DPCDS": soa(dp), "PORO": poro, "POROP": poroP, "ROCKVP": Vp}
    return out, (grid, f, kr, pc, row, key, slot)


def _exact_adjoint(case, seed):
    o, (grid, f, kr, pc, row, key, slot) = _exact_assemble(case, seed)
    nb, nconn, nc = grid.nb, grid.nconn, case["Nc"] + 1
    B = nc + 1
    lam = _lambda(nb * B, seed).reshape(nb, B)
    cb, ce = (torch.as_tensor(a, dtype=torch.int64, device="cuda") for a in (grid.conn_b, grid.conn_e))
    col = torch.cat([torch.arange(nb, device="cuda"), ce, cb])
    val = o["val"].reshape(-1, B, B)
    gX = torch.zeros(nb, B, dtype=torch.float64, device="cuda")
    for lo in range(0, row.numel(), 400000):
        hi = min(row.numel(), lo + 400000)
        gX.index_add_(0, col[lo:hi], (lam[row[lo:hi]][:, None, :] @ val[slot[lo:hi]])[:, 0])
    b, e, dPhi, up, act, _, _, _ = _fluxes(f, grid, kr, pc, 0, nconn)
    gT = torch.zeros(nconn, dtype=torch.float64, device="cuda")
    dl = lam[b, 1:] - lam[e, 1:]
    for j in range(3):
        u = torch.where(up[:, j], b, e)
        m = torch.where(act[:, j], kr[u, j] / f["MU"][u, j] * f["XI"][u, j] * dPhi[:, j], 0.0)
        gT += m * (f["XIJ"][u, j] * dl).sum(1)
    return {"gX": gX.reshape(-1), "gT": DT * gT, "gV": lam[:, 0].contiguous()}


def exact(case, seed):
    """The assembly and the gradients in plain torch.  A flash has no such value: it is defined by the
    iteration path of the reference's algorithm (caps, restarts, the phase labels that follow from them), and the
    solves' systems come out of a flash; both are compared with earlier results alone."""
    if case["kind"] == "assemble":
        return _exact_assemble(case, int(seed))[0]
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, int(seed))
    return None
