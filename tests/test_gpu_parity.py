"""HIP path vs the C oracle on the same inputs (FP64, 1e-10 relative,
identical phase labels).  All compute goes through libocpx.so."""
import numpy as np
import pytest

from opencaeporox_amd import workload as W
from opencaeporox_amd.fim import BATCHED, PLAIN, IsoTFIM
from oracle.oracle import state_from_workload
from tests.conftest import (FLOOR, PARITY_RTOL, SPREAD_MULT, cell_spread, close, degenerate, label_stable,
                            perturbed_oracle_states, rel_err, rounding_spread)

pytestmark = pytest.mark.gpu

FLASH_FIELDS = ["S", "XIJ", "RHO", "XI", "MU", "RHOP", "XIP", "MUP", "RHOX", "XIX", "MUX",
                "NT", "VF", "VFP", "VFI"]
FLASH_OUT = FLASH_FIELDS + ["PHASEEXIST", "DSEC_DPRI"]


def _bits(v):
    return "|".join(str(1 << b) for b in range(10) if (v >> b) & 1) or "0"


def _compare_flash(dev, st, Nc, tag, others, min_cells=0, min_two_phase=0, max_degenerate_flips=0.01):
    """Labels identical on every cell whose labels the oracle reproduces under
    rounding-level perturbations (others: its FMA build, P * (1 + 2^-50)),
    capped trajectories included, unless the trajectory passes through
    degenerate iterates (oracle bits 16, 32): label differences there are
    counted and bounded (max_degenerate_flips of the cells).  Every field within
    PARITY_RTOL on every cell where device and oracle labels agree, or within
    SPREAD_MULT times the oracle's own spread over the cell under those
    perturbations where that is larger.  Prints per field how many entries pass
    only because of the scale floor (FLOOR) and asserts the compared-cell
    counts.  Returns the label-agreeing, label-stable cells."""
    n = dev.nb
    pe_d = dev.get("PHASEEXIST").reshape(n, 3)
    pe_o = st.a["PHASEEXIST"].reshape(n, 3)
    mism = np.any(pe_d != pe_o, axis=1)
    stable = label_stable(st, others)
    deg = degenerate(st.ill)
    bad = np.where(mism & stable & ~deg)[0]
    flips = np.where(mism & stable & deg)[0]
    print(f"{tag}: {stable.sum()} of {n} cells label-stable in the oracle, {(stable & ~deg).sum()} of them "
          f"without degenerate iterates; {mism.sum()} label mismatches: {(mism & ~stable).sum()} in unstable cells, "
          f"{flips.size} in degenerate stable cells (bits {[_bits(int(st.ill[c])) for c in flips[:10]]})")
    assert bad.size == 0, (f"{tag}: labels differ in {bad.size} label-stable cells, "
                           f"e.g. {bad[:10]} with bits {[_bits(int(st.ill[c])) for c in bad[:10]]}")
    assert flips.size <= max_degenerate_flips * n, f"{tag}: {flips.size} label flips in degenerate cells"
    same = ~mism
    fo_d, fo_o = dev.get("FTYPE_OUT"), st.a["FTYPE_OUT"]
    assert np.array_equal(fo_d[same & stable], fo_o[same & stable]), f"{tag}: ftype differs"
    loose = np.zeros(n, bool)
    for f in FLASH_FIELDS + ["DSEC_DPRI"]:
        rowwise = f == "DSEC_DPRI"
        b = st.a[f].reshape(n, -1)
        a = dev.get(f).reshape(n, -1)
        err = np.zeros_like(b)
        err0 = np.zeros_like(b)
        err[same] = rel_err(a[same], b[same], rowwise)
        err0[same] = rel_err(a[same], b[same], rowwise, floor=0.0)
        spread = cell_spread(rounding_spread(st, others, f, n, rowwise))
        spread0 = cell_spread(rounding_spread(st, others, f, n, rowwise, floor=0.0))
        tol = np.maximum(PARITY_RTOL, SPREAD_MULT * spread)
        tol0 = np.maximum(PARITY_RTOL, SPREAD_MULT * spread0)
        over = np.any(err > PARITY_RTOL, axis=1)
        loose |= over
        fail = np.any(err > tol, axis=1)
        floor_only = int(np.sum((err0 > tol0) & (err <= tol)))
        if over.any() or floor_only:
            c = np.where(over)[0]
            print(f"{tag}: {f} above {PARITY_RTOL:g} in {c.size} cells (worst {err.max():.2e}; oracle's own "
                  f"rounding spread there up to {spread[c].max() if c.size else 0:.2e}); {floor_only} entries "
                  f"pass only by the {FLOOR:g} scale floor (worst plain relative {err0.max():.2e})")
        assert not fail.any(), (f"{tag}: {f} differs beyond tolerance in cells {np.where(fail)[0][:8]}: "
                                f"err {err[fail].max():.2e}, spread {spread[fail].max():.2e}")
    two = same & (pe_o[:, 0] > 0) & (pe_o[:, 1] > 0)
    print(f"{tag}: {same.sum()} cells field-compared ({two.sum()} two-phase): "
          f"{same.sum() - loose[same].sum()} within {PARITY_RTOL:g}, "
          f"{loose[same].sum()} within {SPREAD_MULT:g}x the oracle's rounding spread")
    assert same.sum() >= min_cells, f"{tag}: only {same.sum()} cells compared"
    assert two.sum() >= min_two_phase, f"{tag}: only {two.sum()} two-phase cells compared"
    return same & stable & ~deg


@pytest.mark.parametrize("mode,lanes", [(PLAIN, 1), (BATCHED, 1), (BATCHED, 4), (BATCHED, 8)])
def test_flash_config1(oracle, oracle_fma, mode, lanes):
    wl = W.cube_grid()
    dev = IsoTFIM.from_workload(wl)
    dev.set_flash_mapping(lanes)
    st = state_from_workload(wl)
    others = perturbed_oracle_states(oracle, oracle_fma, wl.fluid, st)
    dev.CalFlash(mode)
    oracle.cal_flash(wl.fluid, st)
    # the 202 two-phase cells of this grid all stop Rachford-Rice at its cap in
    # the reference algorithm; they are compared like the others (a few are
    # label-unstable under rounding and may take the other label)
    keep = _compare_flash(dev, st, wl.Nc, f"10x10x10 mode {mode} lanes {lanes}", others,
                          min_cells=980, min_two_phase=195)
    # SkipPSA next-step data
    assert np.array_equal(dev.get("SKIP_FLAG")[keep], st.a["SKIP_FLAG"][keep])
    ok, worst = close(dev.get("SKIP_MINEIG")[keep], st.a["SKIP_MINEIG"][keep], rtol=1e-6)
    assert ok, f"minEig worst {worst}"


# team sizes built per Nc: 4 always, 8 from Nc = 5, 16 from Nc = 9; the
# batched mode with every stage (3), the stability and split-SSM stages (2),
# the stability stages alone (1) and none (0); "long": every stage, on a
# second flash in which the cells over 150 fugacity evaluations in the first
# run on the branch beside the stages; "one lane": every stage with one lane per
# cell, as contexts of many cells run them
PE_CASES = [(Nc, m, lanes, stages) for Nc in (3, 4, 5, 9, 12)
            for m, lanes, stages in ((PLAIN, 1, 0), (BATCHED, 1, 3), (BATCHED, 4, 3), (BATCHED, 8, 3),
                                     (BATCHED, 16, 3), (BATCHED, 4, 2), (BATCHED, 4, 1), (BATCHED, 1, 0),
                                     (BATCHED, 4, 0), (BATCHED, 1, "long"), (BATCHED, 4, "long"),
                                     (BATCHED, 4, "one lane"))
            if lanes < 8 or (lanes == 8 and Nc >= 5) or (lanes == 16 and Nc >= 9)]
# and the team kernels of the other component counts
PE_CASES += [(Nc, BATCHED, lanes, 3) for Nc in (2, 6, 7, 8, 10, 11) for lanes in (4, 8, 16)
             if lanes < 8 or (lanes == 8 and Nc >= 5) or (lanes == 16 and Nc >= 9)]


@pytest.mark.parametrize("Nc,mode,lanes,stages", PE_CASES)
def test_phase_equilibrium_cells(oracle, oracle_fma, Nc, mode, lanes, stages):
    """Phase count, split and flash type per cell against the oracle, for
    the one-cell-per-lane kernels and the team mapping (one component per
    lane), with and without the stability stages."""
    # pressures across both phase regions; seed 44 gives the 3-component
    # fluid a two-phase region there
    wl, z = W.flash_cells(3000, Nc, seed=44 if Nc == 3 else 10 + Nc, P=np.linspace(5.0, 250.0, 3000))
    dev = IsoTFIM.from_workload(wl)
    dev.set_flash_mapping(lanes)
    if stages == "long":
        dev.set_flash_stages(3)
        dev.set_flash_long(0)
        dev.PhaseEquilibrium(mode)
        nlong = int(np.sum(dev.get("ITERS").reshape(-1, 8)[:, 5] > 150))
        print(f"Nc={Nc}: {nlong} cells over 150 evaluations go to the branch")
        assert nlong > 10
        dev.set_flash_long(150)
    elif stages == "one lane":
        dev.set_flash_variants(trials_apart=False, lane_pairs=False)
        assert dev.flash_variants() == (False, False)
    else:
        dev.set_flash_stages(stages)
    dev.PhaseEquilibrium(mode)
    NP, nu, x = dev.pe_result()
    P = wl.state["P"]
    T = wl.state["T"] + W.CONV4
    NPo, nuo, xo, fo, ito = oracle.phase_equilibrium(wl.fluid, P, T, z)
    ill = oracle.last_ill
    runs = [oracle_fma.phase_equilibrium(wl.fluid, P, T, z),
            oracle.phase_equilibrium(wl.fluid, P * (1 + 2.0 ** -50), T, z),
            oracle.phase_equilibrium(wl.fluid, P * (1 - 2.0 ** -50), T, z),
            oracle_fma.phase_equilibrium(wl.fluid, P * (1 - 2.0 ** -50), T, z)]
    # NP must agree wherever the oracle reproduces its own NP under the
    # rounding-level perturbations, capped trajectories included
    stable = np.ones(len(P), bool)
    for r in runs:
        stable &= r[0] == NPo
    mism = NP != NPo
    deg = degenerate(ill)
    print(f"Nc={Nc}: {stable.sum()} of {len(P)} cells NP-stable in the oracle, {mism.sum()} NP mismatches, "
          f"{(mism & stable & deg).sum()} of them in degenerate stable cells")
    bad = np.where(mism & stable & ~deg)[0]
    assert bad.size == 0, f"Nc={Nc}: NP differs in {bad.size} NP-stable cells {bad[:10]}"
    assert (mism & stable & deg).mean() <= 0.01
    assert mism.mean() < 0.02
    two = (NP == 2) & (NPo == 2)
    assert (two & (ill == 0)).sum() > 100, "workload must contain well-conditioned two-phase cells"
    for name, dv, ov, k in (("nu", nu, nuo, 1), ("x", x, xo, 2)):
        dv, ov = dv[two].reshape(two.sum(), -1), ov[two].reshape(two.sum(), -1)
        err = rel_err(dv, ov)
        err0 = rel_err(dv, ov, floor=0.0)
        spread = np.zeros_like(err)
        spread0 = np.zeros_like(err)
        for r in runs:
            same = (r[0] == NPo)[two]
            e = rel_err(r[k][two].reshape(two.sum(), -1), ov)
            e0 = rel_err(r[k][two].reshape(two.sum(), -1), ov, floor=0.0)
            e[~same] = 0
            e0[~same] = 0
            spread = np.maximum(spread, e)
            spread0 = np.maximum(spread0, e0)
        spread, spread0 = cell_spread(spread), cell_spread(spread0)
        tol = np.maximum(PARITY_RTOL, SPREAD_MULT * spread)
        tol0 = np.maximum(PARITY_RTOL, SPREAD_MULT * spread0)
        over = np.any(err > PARITY_RTOL, axis=1)
        print(f"Nc={Nc}: {name} above {PARITY_RTOL:g} in {over.sum()} of {two.sum()} two-phase cells "
              f"(worst {err.max():.2e}, oracle spread there {spread[over].max() if over.any() else 0:.2e}); "
              f"{int(np.sum((err0 > tol0) & (err <= tol)))} entries pass only by the scale floor")
        assert np.all(err <= tol), f"{name}: err {err.max():.2e}"
    keep = stable & ~mism
    assert np.array_equal(dev.get("FTYPE_OUT")[keep], fo[keep])
    # iteration counts agree on clean cells (same algorithm; a converged
    # fixed-point iteration may take one more or one fewer step under
    # different rounding)
    clean = ill == 0
    it = dev.get("ITERS").reshape(-1, 8)
    same = np.mean(np.all(it[clean, :5] == ito[clean, :5], axis=1))
    print(f"iteration counts identical in {100 * same:.1f}% of clean cells")
    assert same > 0.9


def test_batched_equals_plain():
    """The work queue changes the order cells are processed in, nothing else
    (the mapped kernel alone, without the stability stages)."""
    wl, z = W.flash_cells(5000, 9, seed=77)
    a = IsoTFIM.from_workload(wl)
    b = IsoTFIM.from_workload(wl)
    b.set_flash_mapping(1)
    b.set_flash_stages(False)
    a.CalFlash(PLAIN)
    b.CalFlash(BATCHED)
    for f in FLASH_OUT:
        assert np.array_equal(a.get(f), b.get(f), equal_nan=True), f
    ia, ib = a.get("ITERS").reshape(-1, 8), b.get("ITERS").reshape(-1, 8)
    diff = np.any(ia != ib, axis=1)
    if diff.any():
        slots = np.where(np.any(ia != ib, axis=0))[0]
        print(f"ITERS differ in {diff.sum()} cells, slots {slots}, e.g.")
        for c in np.where(diff)[0][:5]:
            print("  ", c, ia[c], ib[c])
    assert diff.mean() < 0.01


def _upload_flash(dev, st):
    for f in FLASH_OUT:
        dev.set(f, st.a[f])


def _compare_assembly(dev, oracle, wl, st, dt, tag):
    dev.CalKrPc()
    dev.CalRock()
    res_d, norms_d = dev.CalRes(dt)
    dev.AssembleMatBulks(dt)
    oracle.cal_krpc(wl.sat, st)
    oracle.cal_rock(wl.rock, st)
    res_o, norms_o = oracle.cal_res(wl.fluid, st, wl.grid, dt)
    rp, col, val = oracle.assemble(wl.fluid, st, wl.grid, dt)
    for f in ["KR", "PC", "PJ", "DKRDS", "DPCDS", "PORO", "POROP", "ROCKVP"]:
        ok, worst = close(dev.get(f), st.a[f])
        assert ok, f"{tag}: {f} worst {worst}"
    ok, worst = close(res_d, res_o)
    assert ok, f"{tag}: resAbs worst {worst}"
    assert norms_d[1] == norms_o[1] and norms_d[3] == norms_o[3]
    ok, worst = close(norms_d[[0, 2]], norms_o[[0, 2]])
    assert ok
    rp_d, col_d, val_d, rhs_d = dev.bsr()
    assert np.array_equal(rp_d, rp) and np.array_equal(col_d, col)
    # each entry relative to itself, floored at FLOOR times the largest entry
    # of its row of the block (one equation's derivatives in one block)
    scale = FLOOR * np.max(np.abs(val), axis=2, keepdims=True)
    err = np.abs(val_d - val) / (np.abs(val) + scale + 1e-300)
    err[val_d == val] = 0
    err0 = np.abs(val_d - val) / (np.abs(val) + 1e-300)
    err0[val_d == val] = 0
    print(f"{tag}: BSR worst {err.max():.2e}; {int(np.sum((err0 > 1e-10) & (err <= 1e-10)))} of {val.size} "
          f"entries pass only by the scale floor (worst plain relative {err0.max():.2e})")
    assert np.max(err) <= 1e-10, (f"{tag}: BSR worst {np.max(err):.3e} at block "
                                  f"{np.unravel_index(np.argmax(err), err.shape)}")
    ok, worst = close(rhs_d, res_o)
    assert ok


def test_assembly_config1_same_flash(oracle):
    """Residual and Jacobian from identical flash outputs: the oracle's flash
    state is uploaded, then kr/Pc, rock, residual and assembly run on the
    device."""
    wl = W.cube_grid()
    st = state_from_workload(wl)
    oracle.cal_flash(wl.fluid, st)
    dev = IsoTFIM.from_workload(wl)
    _upload_flash(dev, st)
    _compare_assembly(dev, oracle, wl, st, 1.0, "10x10x10")


def _clean_grid(seed=31, Nc=3, nx=4, ny=3, nz=2):
    rng = np.random.Generator(np.random.PCG64(seed))
    nb = nx * ny * nz
    k = np.exp(rng.normal(np.log(100.0), 1.0, nb))
    grid = W.cartesian_grid(nx, ny, nz, 6.096, k, k, 0.1 * k, rng.uniform(0.1, 0.3, nb))
    fl = W.make_fluid(Nc, 130)
    rock = W.make_rock()
    stt = W.initial_state(fl, rock, grid, rng.uniform(5.0, 120.0, nb),
                          rng.dirichlet(np.ones(Nc), nb), rng)
    return W.Workload("clean grid", fl, W.make_sat(), rock, grid, stt)


@pytest.mark.parametrize("mode,lanes", [(PLAIN, 1), (BATCHED, 1), (BATCHED, 4)])
def test_newton_passes_end_to_end(oracle, oracle_fma, mode, lanes):
    """Device flash + assembly against the oracle's on a grid whose cells are
    all well-conditioned, then GetSolution and a second pass from the
    two-phase history."""
    wl = _clean_grid()
    dt = 1.0
    dev = IsoTFIM.from_workload(wl)
    dev.set_flash_mapping(lanes)
    st = state_from_workload(wl)
    others = perturbed_oracle_states(oracle, oracle_fma, wl.fluid, st)
    dev.CalFlash(mode)
    oracle.cal_flash(wl.fluid, st)
    assert st.ill.max() == 0
    _compare_flash(dev, st, wl.Nc, "pass1", others, min_cells=dev.nb)
    _compare_assembly(dev, oracle, wl, st, dt, "pass1")
    rng = np.random.Generator(np.random.PCG64(5))
    u = rng.normal(0, 1, dev.nb * dev.bs)
    u.reshape(-1, dev.bs)[:, 0] *= 2.0                        # bar
    u.reshape(-1, dev.bs)[:, 1:] *= 1e-3 * np.abs(st.a["NI"].reshape(-1, dev.nc))
    dev.GetSolution(u, 0.1)
    oracle.get_solution(wl.fluid, st, u, 0.1)
    for f in ["P", "NI", "S", "XIJ"]:
        ok, worst = close(dev.get(f), st.a[f])
        assert ok, f"GetSolution {f} worst {worst}"
    others = perturbed_oracle_states(oracle, oracle_fma, wl.fluid, st)
    dev.CalFlash(mode)
    oracle.cal_flash(wl.fluid, st)
    _compare_flash(dev, st, wl.Nc, "pass2", others, min_cells=dev.nb)
    _compare_assembly(dev, oracle, wl, st, dt, "pass2")


def test_reset_to_last_step_repeats_the_pass():
    """A pass repeated after ResetToLastTimeStep gives the same bits, with the
    long-cell branch routed by the counters saved with the accepted step."""
    wl = W.cube_grid()
    dev = IsoTFIM.from_workload(wl)
    dev.set_flash_long(20)
    dev.newton_pass(1.0, BATCHED)                # the accepted step's flash and counters
    assert np.sum(dev.get("ITERS").reshape(-1, 8)[:, 5] > 20) > 10
    dev.UpdateLastTimeStep()
    dev.newton_pass(1.0, BATCHED)
    ref = [dev.get(f) for f in ("PHASEEXIST", "S", "DSEC_DPRI", "ITERS")] + [dev.bsr()[2]]
    for _ in range(2):
        dev.ResetToLastTimeStep()
        assert np.array_equal(dev.get("NI"), dev.get("LNI"))
        dev.newton_pass(1.0, BATCHED)
        got = [dev.get(f) for f in ("PHASEEXIST", "S", "DSEC_DPRI", "ITERS")] + [dev.bsr()[2]]
        for x, y in zip(got, ref):
            assert np.array_equal(x, y, equal_nan=True)


def test_jt_lambda_dot_product():
    wl = W.cube_grid()
    dev = IsoTFIM.from_workload(wl)
    dev.newton_pass(1.0, BATCHED)
    rp, col, val, _ = dev.bsr()
    rng = np.random.Generator(np.random.PCG64(9))
    n, b = dev.nb, dev.bs
    v = rng.normal(size=n * b)
    lam = rng.normal(size=n * b)
    Jv = np.zeros(n * b)
    for r in range(n):
        for s in range(rp[r], rp[r + 1]):
            Jv[r * b:(r + 1) * b] += val[s] @ v[col[s] * b:(col[s] + 1) * b]
    JTl = dev.jt_lambda(lam)
    assert abs(Jv @ lam - v @ JTl) <= 1e-10 * (abs(Jv @ lam) + np.abs(Jv).dot(np.abs(lam)))


def test_autotuner_picks_a_valid_mapping():
    wl, _ = W.flash_cells(20000, 6, seed=3)
    dev = IsoTFIM.from_workload(wl)
    ms = dev.autotune_flash()
    nat = ms.pop("natural_order")
    assert set(ms) == {1, 4, 8} and all(v > 0 for v in ms.values()) and nat > 0
    assert dev.flash_mapping() == min(ms, key=ms.get)
    assert dev.flash_queue_order() == (ms[dev.flash_mapping()] <= nat)
    dev.set_flash_mapping(0)
    assert dev.flash_mapping() == min(ms, key=ms.get)


@pytest.mark.parametrize("lanes", [1, 8])
def test_queue_order_does_not_change_results(lanes):
    """The longest-first queue only reorders work: a second batched flash
    (ordered by the first one's counts) gives the same bits as a flash in
    natural order."""
    wl, _ = W.flash_cells(20000, 6, seed=11, P=np.linspace(5.0, 250.0, 20000))
    a = IsoTFIM.from_workload(wl)
    b = IsoTFIM.from_workload(wl)
    for d in (a, b):
        d.set_flash_mapping(lanes)
    a.set_flash_queue_order(True)
    b.set_flash_queue_order(False)
    for _ in range(2):
        a.set_state(wl.state)
        b.set_state(wl.state)
        a.CalFlash(BATCHED)
        b.CalFlash(BATCHED)
    for f in ("PHASEEXIST", "S", "XIJ", "DSEC_DPRI", "ITERS"):
        assert np.array_equal(a.get(f), b.get(f)), f
    a.close()
    b.close()


def test_graph_replay_matches_eager():
    """Three graph replays equal three eager passes of the same sequence, bit
    for bit (from the second pass on, the cells that took longest in the
    previous flash run on the flash's second branch)."""
    wl = W.cube_grid()
    a = IsoTFIM.from_workload(wl)
    b = IsoTFIM.from_workload(wl)
    a.set_flash_long(20)
    b.set_flash_long(20)
    for rep in range(3):
        for d, graph in ((a, False), (b, True)):
            d.set_state(wl.state)
            d.set("SKIP_FLAG", np.zeros(d.nb, np.uint32))
            d.newton_pass(1.0, BATCHED, graph=graph)
        if rep:
            assert np.sum(a.get("ITERS").reshape(-1, 8)[:, 5] > 20) > 10
        ref = [a.get(f) for f in ("S", "DSEC_DPRI", "ITERS")] + [a.bsr()[2]]
        got = [b.get(f) for f in ("S", "DSEC_DPRI", "ITERS")] + [b.bsr()[2]]
        for x, y in zip(got, ref):
            assert np.array_equal(x, y), f"replay {rep} differs"
