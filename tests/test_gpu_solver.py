"""Device linear solve (ocpx_linear_solve: ABF decoupling + FGMRES(30) with the
CPR-type preconditioner by default, BiCGStab + block Jacobi as the other
method) against a direct sparse solve of the same system, the reference's
solver settings on the heterogeneous grid with and without its five wells,
and a Newton iteration that stays on the device (assemble -> solve ->
GetSolution)."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from opencaeporox_amd import abi
from opencaeporox_amd import workload as W
from opencaeporox_amd.fim import BATCHED, IsoTFIM

pytestmark = pytest.mark.gpu


def _system(dev):
    rowptr, col, val, rhs = dev.bsr()
    B = dev.bs
    J = sp.bsr_matrix((val.reshape(-1, B, B), col, rowptr), shape=(dev.nb * B, dev.nb * B)).tocsr()
    return J, rhs


@pytest.mark.parametrize("method", [1, 0])
def test_linear_solve_matches_direct_solve(method):
    wl = W.cube_grid()
    dev = IsoTFIM.from_workload(wl)
    dev.set_linear_solver(method)
    dev.newton_pass(1.0, BATCHED)
    J, rhs = _system(dev)
    u, it, rr = dev.LinearSolve(rtol=1e-12, maxit=2000)
    print(f"10x10x10, method {method}: {it} iterations, ||r||/||b|| {rr:.2e}")
    assert it > 0 and rr < 1e-12
    true = np.linalg.norm(rhs - J @ u) / np.linalg.norm(rhs)
    ref = spla.spsolve(J.tocsc(), rhs)
    err = np.linalg.norm(u - ref) / np.linalg.norm(ref)
    print(f"10x10x10: true residual {true:.2e}, |u - u_direct| / |u_direct| {err:.2e}")
    assert true < 1e-11
    # forward error within cond(J) times the residual: cond(J) is about 2e4 here
    assert err < 1e-7
    dev.close()


def test_linear_solve_reference_tolerance_on_heterogeneous_grid():
    # the reference's solver settings (1e-3 on ||r|| / ||b||, 200 iterations)
    wl = W.heterogeneous_grid(20, 20, 10, Nc=6)
    dev = IsoTFIM.from_workload(wl)
    dev.newton_pass(1.0, BATCHED)
    J, rhs = _system(dev)
    u, it, rr = dev.LinearSolve(rtol=1e-3, maxit=200)
    true = np.linalg.norm(rhs - J @ u) / np.linalg.norm(rhs)
    print(f"20x20x10: {it} iterations, recursive {rr:.2e}, true {true:.2e}")
    assert it > 0 and rr < 1e-3
    assert true < 2e-3
    dev.close()


def test_cpr_on_the_heterogeneous_grid_with_wells():
    """The heterogeneous grid (lognormal permeability, sigma = 2, kv/kh =
    0.1) with one composition everywhere: at 20x20x10 with its five vertical
    wells in the system the reference's settings converge, and so they do on
    the full 100x100x50 grid.  (Per-cell random compositions put unrelated
    fluids side by side; their Newton system defeats every preconditioner
    tried, an exact pressure solve included, from 50x50x25 on.)"""
    from opencaeporox_amd import wells as WL
    wl = W.heterogeneous_grid(20, 20, 10, Nc=6, composition="uniform")
    dev = IsoTFIM.from_workload(wl)
    dev.SetWells(WL.corner_and_centre_wells(wl))
    dev.newton_pass(1.0, BATCHED)
    dev.CalResWells(1.0, jacobian=True)
    u, it, rr = dev.LinearSolve(rtol=1e-3, maxit=200)
    print(f"20x20x10 with wells: {it} iterations, decoupled ||r||/||b|| {rr:.2e}")
    assert it > 0 and rr < 1e-3
    assert u.size == (dev.nb + 5) * dev.bs and np.all(np.isfinite(u))
    dev.close()
    wl = W.heterogeneous_grid(100, 100, 50, Nc=6, composition="uniform")
    dev = IsoTFIM.from_workload(wl)
    dev.newton_pass(1.0, BATCHED)
    u, it, rr = dev.LinearSolve(rtol=1e-3, maxit=200, fetch=False)
    print(f"100x100x50: {it} iterations, decoupled ||r||/||b|| {rr:.2e}")
    assert it > 0 and rr < 1e-3
    dev.close()


def test_nonconvergence_is_reported():
    wl = W.heterogeneous_grid(20, 20, 10, Nc=6)
    dev = IsoTFIM.from_workload(wl)
    dev.newton_pass(1.0, BATCHED)
    u, it, rr = dev.LinearSolve(rtol=1e-30, maxit=3)
    assert it == -3 and rr > 1e-30
    # a solve that did not converge leaves nothing to apply: the state is unchanged
    P0 = dev.get("P").copy()
    from opencaeporox_amd.fim import OcpxError
    with pytest.raises(OcpxError, match="needs ocpx_linear_solve"):
        dev.GetSolution(None)
    assert np.array_equal(dev.get("P"), P0)
    # after a converged solve it applies once
    u, it, rr = dev.LinearSolve(rtol=1e-1, maxit=200)
    assert it > 0
    dev.GetSolution(None)
    assert not np.array_equal(dev.get("P"), P0)
    with pytest.raises(OcpxError, match="needs ocpx_linear_solve"):
        dev.GetSolution(None)
    dev.close()


def _smooth_grid(nx=8, ny=8, nz=4, Nc=4, seed=7):
    """A time step a Newton iteration can converge: hydrostatic pressure, one
    composition everywhere, the residual coming from the +-1% Ni and
    +-0.1 MPa perturbation of the previous step.  (The parity configurations'
    random pressure fields give Newton steps of thousands of bar.)"""
    rng = np.random.Generator(np.random.PCG64(seed))
    nb = nx * ny * nz
    kx = np.exp(rng.normal(np.log(100.0), 1.0, nb))
    grid = W.cartesian_grid(nx, ny, nz, 6.096, kx, kx, 0.1 * kx, rng.uniform(0.1, 0.3, nb))
    fl = W.make_fluid(Nc, 107)
    P = 150.0 + 0.0980665 * (grid.depth - grid.depth.min())
    z = np.tile(rng.dirichlet(np.ones(Nc)), (nb, 1))
    st = W.initial_state(fl, W.make_rock(), grid, P, z, rng)
    return W.Workload("smooth", fl, W.make_sat(), W.make_rock(), grid, st)


def test_newton_iterations_on_device():
    """Assemble -> device solve -> device GetSolution, repeated: the residual
    falls quadratically (the oracle with a direct solve goes 4.5e3, 18,
    3e-2, 2.5e-6 on this step), and the device-solution path matches
    GetSolution with the same u handed over from the host."""
    wl = _smooth_grid()
    a = IsoTFIM.from_workload(wl)
    b = IsoTFIM.from_workload(wl)
    norms = []
    for k in range(4):
        a.newton_pass(1.0, BATCHED)
        b.newton_pass(1.0, BATCHED)
        res, nrm = a.CalRes(1.0)
        norms.append(np.abs(res).max())
        u, it, rr = a.LinearSolve(rtol=1e-10, maxit=2000)
        assert it > 0
        a.GetSolution(None, 0.2)
        b.GetSolution(u, 0.2)
        for f in ("P", "NI", "S"):
            assert np.array_equal(a.get(f), b.get(f)), f"iteration {k} field {f}"
    print("max |R| per Newton iteration:", " ".join(f"{v:.3e}" for v in norms))
    assert norms[-1] < 1e-6 * norms[0]
    a.close()
    b.close()


def _odd_cycle(grid, nx):
    """The grid with the extra connection (0, nx + 1): cells 0, 1, nx + 1 form a
    triangle, so the block graph needs three colours."""
    k = int(np.searchsorted(grid.conn_b, 0, side="right"))
    ins = lambda a, v: np.insert(a, k, v)
    return W.Grid(grid.nx, grid.ny, grid.nz, grid.v, grid.depth, grid.poro, ins(grid.conn_b, 0).astype(np.int32),
                  ins(grid.conn_e, nx + 1).astype(np.int32), ins(grid.trans, grid.trans.mean()))


# (Nc, grid, extra connection): fewer rows than the dense coarsest level, one and several levels in one
# workgroup, levels above it, odd block sizes, and a block graph of three colours
@pytest.mark.parametrize("Nc,dims,odd", [(3, (2, 2, 2), False), (5, (4, 4, 4), False), (2, (5, 13, 1), False),
                                         (6, (13, 12, 9), False), (4, (23, 19, 11), False), (3, (7, 6, 5), True),
                                         (6, (16, 9, 8), True)])
def test_cpr_over_grids_and_colours(Nc, dims, odd):
    rng = np.random.Generator(np.random.PCG64(17))
    nx, ny, nz = dims
    nb = nx * ny * nz
    k = np.exp(rng.normal(np.log(100.0), 1.0, nb))
    grid = W.cartesian_grid(nx, ny, nz, 6.096, k, k, 0.1 * k, rng.uniform(0.1, 0.3, nb))
    if odd:
        grid = _odd_cycle(grid, nx)
    fl, rock = W.make_fluid(Nc, 103), W.make_rock()
    z = np.tile(rng.dirichlet(np.ones(Nc)), (nb, 1))
    st = W.initial_state(fl, rock, grid, 200.0 + rng.normal(0, 5.0, nb), z, rng)
    dev = IsoTFIM.from_workload(W.Workload("cpr", fl, W.make_sat(), rock, grid, st))
    dev.newton_pass(0.01, BATCHED)
    J, rhs = _system(dev)
    u, it, rr = dev.LinearSolve(rtol=1e-11, maxit=200)
    u2, it2, _ = dev.LinearSolve(rtol=1e-11, maxit=200)
    assert it > 0 and rr < 1e-11
    assert it2 == it and np.array_equal(u, u2), "the solve is not repeatable"
    true = np.linalg.norm(rhs - J @ u) / np.linalg.norm(rhs)
    ref = spla.spsolve(J.tocsc(), rhs)
    err = np.linalg.norm(u - ref) / np.linalg.norm(ref)
    print(f"{dims} Nc={Nc} odd={odd}: {it} iterations, true {true:.2e}, error {err:.2e}")
    # 1e-11 on the decoupled residual, cond(J) below 1e5: as the direct-solve test above
    assert true < 1e-9 and err < 1e-6
    dev.close()


def test_solve_after_new_transmissibilities_on_a_callers_stream():
    """New transmissibilities rebuild the pressure hierarchy of a context whose
    other buffers are in place; on a stream that is not ordered with the default
    one the solve is that of a fresh context, bit for bit."""
    rng = np.random.Generator(np.random.PCG64(29))
    nx, ny, nz, Nc = 23, 19, 11, 4
    nb = nx * ny * nz
    k = np.exp(rng.normal(np.log(100.0), 1.0, nb))
    grid = W.cartesian_grid(nx, ny, nz, 6.096, k, k, 0.1 * k, rng.uniform(0.1, 0.3, nb))
    fl, rock = W.make_fluid(Nc, 103), W.make_rock()
    z = np.tile(rng.dirichlet(np.ones(Nc)), (nb, 1))
    st = W.initial_state(fl, rock, grid, 200.0 + rng.normal(0, 5.0, nb), z, rng)
    wl = W.Workload("cpr", fl, W.make_sat(), rock, grid, st)
    stream = C.c_void_p()
    assert abi.load().hipStreamCreateWithFlags(C.byref(stream), 1) == 0        # hipStreamNonBlocking
    dev = IsoTFIM.from_workload(wl, stream=stream)
    dev.UpdateLastTimeStep()
    T = grid.trans
    for trans in (T, T * rng.uniform(0.1, 10.0, T.size), T * rng.uniform(0.01, 1.0, T.size)):
        dev.set_geometry(trans=trans)
        dev.ResetToLastTimeStep()
        dev.newton_pass(0.01, BATCHED)
        u, it, rr = dev.LinearSolve(rtol=1e-10, maxit=200)
        fresh = IsoTFIM.from_workload(wl)
        fresh.set_geometry(trans=trans)
        fresh.UpdateLastTimeStep()
        fresh.newton_pass(0.01, BATCHED)
        v, jt, _ = fresh.LinearSolve(rtol=1e-10, maxit=200)
        assert it == jt > 0 and rr < 1e-10
        assert np.array_equal(u, v)
        fresh.close()
    dev.close()
    assert abi.load().hipStreamDestroy(stream) == 0


def _cpr_case(Nc, dims, sigma, odd=False):
    rng = np.random.Generator(np.random.PCG64(17))
    nx, ny, nz = dims
    nb = nx * ny * nz
    k = np.exp(rng.normal(np.log(100.0), sigma, nb))
    grid = W.cartesian_grid(nx, ny, nz, 6.096, k, k, 0.1 * k, rng.uniform(0.1, 0.3, nb))
    if odd:
        grid = _odd_cycle(grid, nx)
    fl, rock = W.make_fluid(Nc, 103), W.make_rock()
    z = np.tile(rng.dirichlet(np.ones(Nc)), (nb, 1))
    st = W.initial_state(fl, rock, grid, 200.0 + rng.normal(0, 5.0, nb), z, rng)
    return W.Workload("cpr", fl, W.make_sat(), rock, grid, st)


def _decoupled_residual(D, J, rhs, u):
    """||D^-1 (rhs - J u)|| / ||D^-1 rhs|| with the diagonal blocks D."""
    b = D.shape[1]
    solve = lambda v: np.linalg.solve(D, v.reshape(-1, b, 1)).ravel()
    return np.linalg.norm(solve(rhs - J @ u)) / np.linalg.norm(solve(rhs))


def test_cpr_on_long_vectors_past_a_restart():
    """Vectors of more than 1,048,576 entries, no multiple of a tile, over more than the 30 iterations to a
    restart: the basis kernels of long vectors at every number of basis vectors, checked on the host."""
    wl = _cpr_case(6, (61, 57, 43), 2.0)
    dev = IsoTFIM.from_workload(wl)
    dev.newton_pass(0.01, BATCHED)
    assert dev.nb * dev.bs > 512 * 256 * 8 and dev.nb * dev.bs % 2048
    J, rhs = _system(dev)
    rp, _, val, _ = dev.bsr()
    u, it, rr = dev.LinearSolve(rtol=1e-11, maxit=200)
    res = _decoupled_residual(val[rp[:-1]], J, rhs, u)
    print(f"61x57x43: {it} iterations, decoupled residual {rr:.2e}, on the host {res:.2e}")
    assert it > 30 and rr < 1e-11
    # the device stops on its own value of this residual; the host's differs by rounding
    assert res < 2e-11
    dev.close()


@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("Nc,dims", [(3, (7, 6, 5)), (6, (16, 9, 8))])
def test_cpr_with_wells_over_colours(Nc, dims, odd):
    """The wells' rows beside both sweeps, the two-coloured one and the one for any number of colours."""
    from opencaeporox_amd import wells as WL
    wl = _cpr_case(Nc, dims, 1.0, odd)
    wells = WL.corner_and_centre_wells(wl)
    dev = IsoTFIM.from_workload(wl)
    dev.SetWells(wells)
    dev.newton_pass(0.01, BATCHED)
    _, wres = dev.CalResWells(0.01, jacobian=True)
    rp, col, val, rhs = dev.bsr()
    J, f = WL.full_system(rp, col, val, rhs, wells, *dev.well_blocks(), wres, dev.bs)
    u, it, rr = dev.LinearSolve(rtol=1e-11, maxit=200)
    true = np.linalg.norm(f - J @ u) / np.linalg.norm(f)
    ref = spla.spsolve(J.tocsc(), f)
    err = np.linalg.norm(u - ref) / np.linalg.norm(ref)
    print(f"{dims} Nc={Nc} odd={odd} with wells: {it} iterations, true {true:.2e}, error {err:.2e}")
    assert it > 0 and rr < 1e-11
    # as test_cpr_over_grids_and_colours
    assert true < 1e-9 and err < 1e-6
    dev.close()


@pytest.mark.parametrize("odd", [False, True])
def test_cpr_with_ill_conditioned_diagonal_blocks(odd):
    """The rows of a tenth of the cells multiplied by matrices of condition 1e8: the decoupled system is the
    same, the diagonal blocks are not.  Both sweeps solve it as before; the inverse of such a block is
    off by 1e-16 times its condition, of which little reaches the residual (1e-8 of it here)."""
    dev = IsoTFIM.from_workload(_cpr_case(6, (13, 12, 9), 1.0, odd))
    dev.newton_pass(0.01, BATCHED)
    J, rhs = _system(dev)
    rp, _, val, _ = dev.bsr()
    b, nb = dev.bs, dev.nb
    D = val[rp[:-1]]
    _, it0, _ = dev.LinearSolve(rtol=1e-6, maxit=200)
    rng = np.random.Generator(np.random.PCG64(3))
    rhs1, val1 = rhs.reshape(nb, b).copy(), val.copy()
    for n in rng.choice(nb, nb // 10, replace=False):
        q, r = (np.linalg.qr(rng.normal(size=(b, b)))[0] for _ in range(2))
        S = (q * np.logspace(0, -8, b)) @ r
        rhs1[n] = S @ rhs1[n]
        val1[rp[n]:rp[n + 1]] = S @ val1[rp[n]:rp[n + 1]]
    lib = abi.load()
    ptr = [C.c_void_p() for _ in range(4)]
    assert lib.ocpx_bsr_device_ptrs(dev.h, *[C.byref(p) for p in ptr]) == 0
    dev.sync()
    for p, a in ((ptr[2], val1), (ptr[3], rhs1)):
        assert lib.hipMemcpy(p, C.c_void_p(a.ctypes.data), C.c_size_t(a.nbytes), C.c_int(1)) == 0
    u, it, rr = dev.LinearSolve(rtol=1e-6, maxit=200)
    res = _decoupled_residual(D, J, rhs, u)
    print(f"odd={odd}: {it0} iterations, {it} with ill-conditioned blocks, residual {rr:.2e}, {res:.2e}")
    assert 0 < it <= it0 + 1 and rr < 1e-6 and res < 2e-6
    dev.close()
