"""Held entries that release, CPML entries, carriers and exits in tiles of many
entries: every particle of the event and held cases stands for K copies of a
K-th of its charge and mass, so that the oracle's run of the few originals
gives the fields, the copies' states and the counters of the many.

FP64: several chunks a tile. FP32-split from 2^19, 2^20 and 2^21 entries on:
chunks of 512, 1024 and 2048 entries, several a lane, and the verifying
residual summed over a lane's entries. Tolerances: FP64 1e-12 as the cases
themselves (K copies of q / K add up to q within a rounding a copy); FP32-split
2e-5 as the cases themselves.
"""
import numpy as np
import pytest

import event_cases as E
import harness as H
from test_gpu_events import SHAPES, rel_l2

pytestmark = pytest.mark.gpu

# (a quarter of the event case's entries leaves within its steps)
FORMS = [("fp64", 20_000), ("fp32-split", 700_000), ("fp32-split", 1_400_000), ("fp32-split", 2_800_000)]


def copies(x, u, q, m, ids, entries):
    """At least `entries` entries: the particles K times over, and K. The copies
    of particle i have the ids (i - 1) K + 1 .. i K."""
    k = entries // len(q) + 1
    number = np.concatenate([(ids - np.uint64(1)) * np.uint64(k) + np.uint64(r + 1) for r in range(k)])
    return (np.tile(x, (k, 1)), np.tile(u, (k, 1)), np.tile(q / k, k), np.tile(m / k, k), number), k


def device(shape, precision, orc, parts, exit_z=float("inf")):
    import aprl_amd as A
    gpu = A.EBFieldGrid(A.EBGridGeometry(*E.DIMS, E.DX, E.DX, E.DZ, E.DZ / H.C_SI), precision=precision)
    win = A.MovingWindowFields(gpu, A.EBCPMLParameters(E.CELLS))
    for a in range(9):
        gpu.set_component(a, orc.view(a))
    cg = A.ConservativeSourceCoupling(gpu, SHAPES[shape][2])
    cg.setFrame(E.GAMMA_BOOST)
    cg.setParticleBoundary(E.CELLS, exit_z)
    if precision != "fp64":
        cg.setSplitTrials(3, True)
    x, u, q, m, ids = parts
    store = A.ParticleStore(gpu, len(q))
    store.upload(x, u, q, m, np.ones(len(q)), ids)
    return gpu, win, cg, store


def run(orc, co, gpu, win, cg, store, steps, exit_z=None):
    rng = np.random.default_rng(4)
    offset = E.OFFSET0
    reports = []
    for n in range(steps):
        print(f"crowded step {n}", flush=True)
        origin = E.window_origin(offset)
        if n:
            co.finish_window(origin)
        lower, inlet, shift = E.planes_for(rng, range(3)), E.planes_for(rng, range(2)), E.planes_for(rng, range(6))
        t = n * E.DZ / H.C_SI
        orc.clear_current(); gpu.clearCurrent()
        orc.window_begin(n, offset, lower); win.beginStep(n, offset, lower)
        orc.window_advance_magnetic(); gpu.advanceMagnetic()
        orc.window_set_inlet(offset, n + 1, *inlet); win.setInlet(*inlet)
        ro = co.step(origin, t, 1) if exit_z is None else co.step(origin, t, 1, exit_z)
        reports.append((ro[0], *cg.step(store, origin, t)))
        offset -= 1
        orc.window_shift(n + 1, offset, shift); win.shift(n + 1, offset, shift)
    return reports


def compare(orc, co, gpu, store, k, tol):
    """Fields, and every copy against its particle of the oracle; returns the
    states in id order."""
    for a in range(9):
        err = rel_l2(gpu.component(a), orc.view(a))
        assert err <= tol, f"component {a}: rel L2 {err:.3e}"
    x, u, _, _, _, ids = store.download()
    states = store.states()
    live = states != 1
    order = np.argsort(ids[live])
    original = (ids[live][order] - 1) // np.uint64(k) + 1
    xo, uo = co.particles()
    oo = np.argsort(co.ids())
    assert np.array_equal(original, np.repeat(np.sort(co.ids()), k))
    ref = np.repeat(xo[oo], k, axis=0)
    assert rel_l2(x[live][order] - ref.mean(0), ref - ref.mean(0)) <= tol
    assert rel_l2(u[live][order], np.repeat(uo[oo], k, axis=0)) <= tol
    return states[live][order]


@pytest.mark.parametrize("shape", ["binomial3", "quintic"])
@pytest.mark.parametrize("precision,entries", FORMS)
def test_crowded_events(precision, entries, shape):
    orc, co = E.oracle_case("orc", SHAPES[shape][0], SHAPES[shape][1], True)
    parts, k = copies(*E.particles(exit_plane=True), entries)
    case = device(shape, precision, orc, parts, E.exit_lab_z())
    reports = run(orc, co, *case, 5, E.exit_lab_z())
    gpu, win, cg, store = case
    tol = 1e-12 if precision == "fp64" else 2e-5
    if precision == "fp64":
        assert all(r[0] == r[1] for r in reports), reports
    assert cg.last_chunks > cg.last_tiles if precision == "fp64" else cg.last_chunks < len(store) / 256
    compare(orc, co, gpu, store, k, tol)
    carriers = store.states() == 1
    *_, idc = co.carriers()
    got = np.sort((store.download()[5][carriers] - 1) // np.uint64(k) + 1)
    assert np.array_equal(got, np.repeat(np.sort(idc), k))
    (counts, charge), (counts_g, charge_g) = co.counters(), cg.boundaryCounters()
    assert np.array_equal(np.asarray(counts) * k, counts_g)
    assert rel_l2(charge_g, charge) <= max(tol, 1e-11)  # k additions of q / k
    assert counts[0] > 0 and counts[18] > 0


@pytest.mark.parametrize("shape", ["binomial3", "quintic"])
@pytest.mark.parametrize("precision,entries", FORMS)
def test_crowded_held(precision, entries, shape):
    orc, co = E.held_oracle_case("orc", SHAPES[shape][0], SHAPES[shape][1])
    x, u, q, m, ids, frozen, beta = E.held_particles()
    parts, k = copies(x, u, q, m, ids, entries)
    case = device(shape, precision, orc, parts)
    gpu, win, cg, store = case
    cg.setActivationPlane(E.activation_lab_z())
    store.setHeld(np.tile(frozen, k), np.tile(beta, k))
    reports = run(orc, co, *case, 5)
    if precision == "fp64":
        assert all(r[0] == r[1] for r in reports), reports
    states = compare(orc, co, gpu, store, k, 1e-12 if precision == "fp64" else 2e-5)
    held = co.frozen()[np.argsort(co.ids())]
    assert np.array_equal((states == 2).astype(np.int32), np.repeat(held, k))
    assert 0 < held.sum() < frozen.sum()  # some released, some still held


@pytest.mark.parametrize("shape", ["binomial3", "quintic"])
def test_crowded_residual(shape):
    """Force and work of the verifying residual, chunks of several entries a lane
    against one: the largest force, and sums whose ratio the copies leave as it
    is. Charges 1e4 times the case's, so that the residual of two trials lies far
    above the FP32 fields' rounding."""
    orc, co = E.held_oracle_case("orc", SHAPES[shape][0], SHAPES[shape][1])
    x, u, q, m, ids, frozen, beta = E.held_particles()
    reports = []
    for entries in (0, 2 ** 19):
        parts, k = copies(x, u, 1e4 * q, 1e4 * m, ids, entries)
        gpu, win, cg, store = device(shape, "fp32-split", orc, parts)
        cg.setSplitTrials(2, True)
        cg.setActivationPlane(E.activation_lab_z())
        store.setHeld(np.tile(frozen, k), np.tile(beta, k))
        print(f"residual of {len(store)} entries", flush=True)
        gpu.clearCurrent()
        win.beginStep(0, E.OFFSET0)
        gpu.advanceMagnetic()
        win.setInlet()
        reports.append(cg.step(store, E.window_origin(E.OFFSET0), 0.0))
    print(reports)
    assert reports[0][1] > 1e-9 and reports[0][2] > 1e-9
    assert np.allclose(reports[0][1:], reports[1][1:], rtol=1e-3, atol=0.0)
