"""Edge cases of the device path against the oracle: the smallest and
largest component counts the kernels are built for, a single cell without
connections, and a grid without cells."""
import ctypes as C

import numpy as np
import pytest

from opencaeporox_amd import abi
from opencaeporox_amd import workload as W
from opencaeporox_amd.fim import BATCHED, PLAIN, IsoTFIM
from oracle.oracle import state_from_workload
from tests.conftest import close, perturbed_oracle_states
from tests.test_gpu_parity import _clean_grid, _compare_assembly, _compare_flash, _upload_flash

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nc,mode,lanes", [(2, PLAIN, 1), (2, BATCHED, 4), (12, BATCHED, 1), (12, BATCHED, 16)])
def test_component_count_extremes(oracle, oracle_fma, Nc, mode, lanes):
    wl = _clean_grid(seed=40 + Nc, Nc=Nc, nx=3, ny=2, nz=2)
    dev = IsoTFIM.from_workload(wl)
    dev.set_flash_mapping(lanes)
    st = state_from_workload(wl)
    others = perturbed_oracle_states(oracle, oracle_fma, wl.fluid, st)
    dev.CalFlash(mode)
    oracle.cal_flash(wl.fluid, st)
    _compare_flash(dev, st, wl.Nc, f"Nc={Nc}", others)
    _upload_flash(dev, st)                       # assembly from identical flash outputs
    _compare_assembly(dev, oracle, wl, st, 1.0, f"Nc={Nc}")
    dev.close()


def _cells(nb, Nc=6, seed=3):
    rng = np.random.Generator(np.random.PCG64(seed))
    g = W.Grid(nb, 1, 1, np.full(nb, 226.5), np.full(nb, 2000.0), np.full(nb, 0.2),
               np.zeros(0, np.int32), np.zeros(0, np.int32), np.zeros(0))
    fl = W.make_fluid(Nc, 100 + seed)
    z = rng.dirichlet(np.ones(Nc), nb) if nb else np.zeros((0, Nc))
    st = W.initial_state(fl, W.make_rock(), g, np.full(nb, 150.0), z, rng)
    return W.Workload(f"{nb} cells", fl, W.make_sat(), W.make_rock(), g, st)


def test_single_cell_without_connections(oracle):
    wl = _cells(1)
    dev = IsoTFIM.from_workload(wl)
    st = state_from_workload(wl)
    dev.CalFlash(BATCHED)
    oracle.cal_flash(wl.fluid, st)
    for f in ("PHASEEXIST", "S", "XIJ", "DSEC_DPRI"):
        ok, worst = close(dev.get(f), st.a[f])
        assert ok, f"{f} worst {worst}"
    _upload_flash(dev, st)
    _compare_assembly(dev, oracle, wl, st, 1.0, "one cell")
    rp, col, val, rhs = dev.bsr()
    assert rp.tolist() == [0, 1] and col.tolist() == [0]
    u, it, rr = dev.LinearSolve(rtol=1e-12, maxit=50)
    assert it > 0
    ref = np.linalg.solve(val[0].reshape(dev.bs, dev.bs), rhs)
    assert np.allclose(u, ref, rtol=1e-10, atol=1e-12 * np.abs(ref).max())
    dev.close()


def test_empty_grid_is_rejected():
    """A context needs at least one cell; creation fails with a message
    instead of a context whose kernels have nothing to launch."""
    from opencaeporox_amd.fim import OcpxError
    wl = _cells(0)
    with pytest.raises(OcpxError, match="no cells"):
        IsoTFIM.from_workload(wl)


# 1,024 workgroups of the residual kernel, one more, and more than the first
# reduction's threads; the largest term in the first, a middle or the last cell
@pytest.mark.parametrize("Nc,nb", [(2, 16384), (6, 8193), (12, 4097), (12, 131077)])
def test_residual_norms_over_many_workgroups(Nc, nb):
    wl = _cells(nb, Nc)
    dev = IsoTFIM.from_workload(wl)
    dev.CalFlash(BATCHED)
    dev.CalKrPc()
    dev.CalRock()
    for n in (0, nb // 2, nb - 1):
        lni = wl.state["LNI"].copy().reshape(nb, dev.nc)
        lni[n] *= 1e4
        dev.set("LNI", lni)
        res, (v, iv, w, iw) = dev.CalRes(1.0)
        r = np.abs(res.reshape(nb, dev.bs))
        rv = (r / dev.get("ROCKVP")[:, None]).max(axis=1)
        rn = (r[:, 1:] / dev.get("NT")[:, None]).max(axis=1)
        assert (iv, iw) == (np.argmax(rv), np.argmax(rn)) and iv == n
        assert np.isclose(v, rv.max(), rtol=1e-14, atol=0) and np.isclose(w, rn.max(), rtol=1e-14, atol=0)
    dev.close()


@pytest.mark.parametrize("Nc", [2, 6, 12])
def test_assembly_with_some_composition_derivatives_zero(oracle, Nc):
    """Phases whose dx_ij/dX are all zero, or all but one entry, beside whole ones."""
    wl = _clean_grid(seed=50 + Nc, Nc=Nc, nx=5, ny=3, nz=3)
    dev = IsoTFIM.from_workload(wl)
    st = state_from_workload(wl)
    oracle.cal_flash(wl.fluid, st)
    nc, b = dev.nc, dev.bs
    rng = np.random.Generator(np.random.PCG64(Nc))
    X = st.a["DSEC_DPRI"].reshape(dev.nb, -1, b)
    dx = X[:, 3:3 + 3 * nc].reshape(dev.nb, 3, nc, b)
    kind = rng.integers(0, 3, (dev.nb, 3))
    one = np.zeros_like(dx)
    one[..., nc - 1, b - 1] = 1e-3
    one[..., 0, 0] = np.where(kind == 1, 0.0, 1e-3)
    dx[:] = np.where((kind == 0)[..., None, None], 0.0, np.where((kind == 1)[..., None, None], one, dx))
    X[:, 3:3 + 3 * nc] = dx.reshape(dev.nb, 3 * nc, b)
    st.a["DSEC_DPRI"] = X.reshape(st.a["DSEC_DPRI"].shape)
    _upload_flash(dev, st)
    _compare_assembly(dev, oracle, wl, st, 1.0, f"Nc={Nc}")
    dev.close()


def _repeated(Nc, m, nb):
    """The first m of 1,501 flash cells, repeated to nb of them."""
    wl, _ = W.flash_cells(1501, Nc, seed=44 if Nc == 3 else 10 + Nc, P=np.linspace(5.0, 250.0, 1501))
    pick = lambda a: np.ascontiguousarray(np.asarray(a).reshape(1501, -1)[np.arange(nb) % m]).ravel()
    g = wl.grid
    grid = W.Grid(nb, 1, 1, pick(g.v), pick(g.depth), pick(g.poro), np.zeros(0, np.int32), np.zeros(0, np.int32),
                  np.zeros(0))
    return W.Workload(wl.name, wl.fluid, wl.sat, wl.rock, grid, {k: pick(a) for k, a in wl.state.items()})


# a few cells, and the last and the first number of cells on either side of the rules for the trials' lanes
# and the pairs of lanes, on 256 compute units of two wavefronts per SIMD
@pytest.mark.parametrize("Nc,nb,variants", [(8, 5, (True, True)), (8, 49152, (True, True)), (8, 49153, (False, True)),
                                            (3, 49153, (False, True)), (3, 655360, (False, True)),
                                            (3, 660001, (False, False)), (8, 655361, (False, False))])
def test_flash_does_not_depend_on_the_number_of_cells(Nc, nb, variants):
    """The same cells, repeated to nb of them, give the same bits however the stages share them out."""
    m = 1501
    out = []
    for n in (m, nb):
        dev = IsoTFIM.from_workload(_repeated(Nc, m, n))
        assert dev.flash_variants() == (variants if n == nb else (True, True))
        dev.CalFlash(BATCHED)
        out.append({f: dev.get(f).reshape(n, -1) for f in ("ITERS", "PHASEEXIST", "S", "XIJ", "FTYPE_OUT")})
        dev.close()
    assert 0 < np.sum(out[0]["PHASEEXIST"][:, :2].sum(axis=1) == 2) < m
    for f in out[0]:
        assert np.array_equal(out[1][f], out[0][f][np.arange(nb) % m]), f


@pytest.mark.parametrize("several", [False, True])
@pytest.mark.parametrize("Nc", range(2, 13))
def test_flash_stage_variants_give_the_same_bits(Nc, several):
    """Every way the stages share their work out, over all component counts, in
    contexts of one model and of several, on the first flash and on the one that
    follows from its phases (the other flash types and the relaxed test)."""
    n = 6000
    out = []
    for apart, pairs in ((False, False), (False, True), (True, False), (True, True)):
        if several:
            dev = IsoTFIM.from_workloads([W.flash_cells(n // 3, Nc, seed=s, P=np.linspace(5.0, 250.0, n // 3))[0]
                                          for s in (44 if Nc == 3 else 10 + Nc, 103, 127)])
        else:
            dev = IsoTFIM.from_workload(W.flash_cells(n, Nc, seed=44 if Nc == 3 else 10 + Nc,
                                                      P=np.linspace(5.0, 250.0, n))[0])
        dev.set_flash_variants(trials_apart=apart, lane_pairs=pairs)
        assert dev.flash_variants() == (apart, pairs)
        got = {}
        for k in range(2):
            dev.CalFlash(BATCHED)
            got.update({(f, k): dev.get(f) for f in ("ITERS", "PHASEEXIST", "S", "XIJ", "FTYPE_OUT", "DSEC_DPRI")})
            got.update({(f, k): a for f, a in zip(("NP", "nu", "x"), dev.pe_result())})
        dev.close()
        out.append(got)
    it = out[0]["ITERS", 0].reshape(-1, 8)
    print(f"Nc={Nc}: {np.sum(it[:, 2] > 0)} cells split, {np.sum(it[:, 3] > 0)} with Newton steps")
    assert np.sum(it[:, 3] > 0) > 100
    bad = []
    for v, got in enumerate(out[1:], 1):
        for f in got:
            if not np.array_equal(got[f], out[0][f], equal_nan=True):
                cells = np.any((got[f] != out[0][f]).reshape(n, -1), axis=1)
                bad.append(f"variant {v} {f}: {np.sum(cells)} cells, first {np.where(cells)[0][:5]}")
    assert not bad, "\n".join(bad)


# one cell, less and more than a wavefront, and one cell more or less than the lanes of a dealt queue can hold
@pytest.mark.parametrize("nb", [1, 63, 65, 1023, 1025, 2049, 5003])
def test_one_lane_kernel_takes_every_cell_once(nb):
    """The one-lane kernel deals a short queue out over its wavefronts; the order
    changes no bits, on the first flash and in longest-first order on the next."""
    wl = _repeated(6, 1501, nb)
    ctx = []
    for mode, longest in ((PLAIN, False), (BATCHED, False), (BATCHED, True)):
        dev = IsoTFIM.from_workload(wl)
        dev.set_flash_mapping(1)
        dev.set_flash_stages(False)
        dev.set_flash_queue_order(longest)
        dev.UpdateLastTimeStep()
        ctx.append((dev, mode))
    for k in range(2):
        out = []
        for dev, mode in ctx:
            dev.CalFlash(mode)
            out.append([dev.get(f) for f in ("FTYPE_OUT", "PHASEEXIST", "S", "XIJ", "DSEC_DPRI")])
        for o in out[1:]:
            assert all(np.array_equal(a, b, equal_nan=True) for a, b in zip(o, out[0])), k
        P = ctx[0][0].get("P")
        for dev, _ in ctx:
            dev.set("P", np.round(P * 1.01, 3))
    for dev, _ in ctx:
        dev.close()


@pytest.mark.parametrize("nb", [1, 64, 30000])
def test_new_context_on_a_stream_not_ordered_with_the_default_one(nb):
    """New buffers are zeroed before anything else reaches them: what is uploaded
    at creation, the first saved time step, the first flash's lists, the wells."""
    from opencaeporox_amd import wells as WL
    stream = C.c_void_p()
    assert abi.load().hipStreamCreateWithFlags(C.byref(stream), 1) == 0        # hipStreamNonBlocking
    wl = _repeated(6, 1501, nb)
    wells = [WL.PeacemanWell("P", WL.PROD, WL.BHP, bhp=1.0, target=1.0, cells=[nb // 2], WI=[2.0])]
    out = []
    for st in (None, stream):
        dev = IsoTFIM.from_workload(wl, stream=st)
        dev.UpdateLastTimeStep()
        got = {f: dev.get(f) for f in ("P", "NI", "FTYPE_IN", "DSEC_DPRI")}
        dev.CalFlash(BATCHED)
        dev.SetWells(wells)
        dev.CalKrPc()
        dev.CalRock()
        dev.AssembleMatBulks(1.0)
        got["norms"], got["wres"] = dev.CalResWells(1.0, jacobian=True)
        for f in ("ITERS", "PHASEEXIST", "XIJ", "DSEC_DPRI"):
            got[f + " after"] = dev.get(f)
        dev.ResetToLastTimeStep()
        got.update({f + " reset": dev.get(f) for f in ("P", "NI", "XIJ", "ITERS")})
        dev.close()
        out.append(got)
    for f in out[0]:
        assert np.array_equal(out[0][f], out[1][f], equal_nan=True), f
    assert np.any(out[0]["P reset"] > 0) and np.any(out[0]["ITERS after"] > 0)
    assert abi.load().hipStreamDestroy(stream) == 0
