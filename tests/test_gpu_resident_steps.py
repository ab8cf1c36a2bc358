"""A micro-step is one evaluation and one update of every running walker,
however the steps are launched: a number of steps leaves every search in the
same state, bit for bit, in chunks of any length, replayed from a graph or
not, timed or not, alone or among walkers that the resident kernel does not
take."""
import numpy as np
import pytest

from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
CU = W.SC_CU


def _field():
    from akmc_amd import lib as L
    return L, L.Field(L.sc_potentials_text([("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])], 2 * CU["a"]))


@pytest.fixture(scope="module")
def searches():
    """relaxed cells and the starts of their searches"""
    L, f = _field()
    cells = [W.sc_cell(n, 5, 6, n_vac=1, jitter=0.01, seed=n) for n in (4, 5, 6, 7)]
    b = L.Batch(f, cells)
    b.start_relax(L.relax_defaults())
    b.run(5000, sync_every=100)
    cells = [W.Cell(p, c.types, c.lat, vacancies=c.vacancies) for p, c in zip(b.positions(), cells)]
    frozen, modes, x0 = [], [], []
    for w, c in enumerate(cells):
        frozen.append((W.site_distances(c, c.vacancies[0]) >= 6.0).astype(np.int32))
        disp, mode = W.local_displacement(c, W.neighbours_of_site(c, c.vacancies[0], 12), 0.1, 11 + w)
        modes.append(mode)
        x0.append(c.pos + disp)
    return cells, (frozen, modes, x0)


def _search(searches, steps, sync, graphs=True, timer=False, extra=None):
    L, f = _field()
    cells, starts = searches
    frozen, modes, x0 = [list(v) for v in starts]
    if extra is not None:
        cells = cells + [extra]
        frozen.append(np.zeros(extra.n, np.int32))  # every atom free: on the chain
        modes.append(np.random.default_rng(3).standard_normal((3, extra.n)))
        x0.append(extra.pos)
    b = L.Batch(f, cells)
    b.set_graphs(graphs)
    b.kernel_timer(timer)
    b.set_basins()
    b.set_basin2(L.basin2_defaults())
    b.set_verify(16, 0.01)
    b.start_dimer(modes, params=L.dimer_defaults(maxParIter=400), x0_per_walker=x0, frozen_per_walker=frozen)
    b.run(steps, sync_every=sync)
    n = len(starts[0])
    return b.status_array()[:n], b.positions()[:n], b.zone()[2][:n]


def test_steps_are_steps(searches):
    kinds = set()
    for steps in (100, 200, 250, 300, 350, 400, 500):
        st, pos, flags = _search(searches, steps, steps)
        assert (flags & 16).all()
        kinds |= set(st["kind"][st["done"] == 0].tolist())
        assert (st["force_calls"][st["done"] == 0] == steps).all()
        print(steps, "done", st["done"].tolist(), "verified", st["verified"].tolist(), "kind", st["kind"].tolist(),
              "force calls", st["force_calls"].tolist(), flush=True)
        for kw in (dict(sync=7), dict(sync=steps, graphs=False), dict(sync=50, timer=True),
                   dict(sync=13, extra=W.sc_cell(4, 4, 4, n_vac=1, jitter=0.01, seed=1))):
            st2, pos2, _ = _search(searches, steps, **kw)
            for k in st.dtype.names:
                assert np.array_equal(st[k], st2[k], equal_nan=True), (steps, kw, k)
            for a, b in zip(pos, pos2):
                assert np.array_equal(a, b), (steps, kw)
    assert len(kinds) > 1 and (st["verified"] == 1).any()  # searches caught in their verification too


def test_verification_turned_on_under_running_searches(searches):
    """The FP64 fixed parts follow with the next chunk: the same bits, step by
    step, as with verification on from the start."""
    L, f = _field()
    cells, (frozen, modes, x0) = searches
    out = []
    for late in (False, True):
        b = L.Batch(f, cells)
        if not late:
            b.set_verify(16, 0.01)
        b.start_dimer(modes, params=L.dimer_defaults(maxParIter=400), x0_per_walker=x0, frozen_per_walker=frozen)
        b.run(100, sync_every=25)
        assert (b.zone()[2] == (21 if late else 17)).all()  # the FP64 parts are pending
        if late:
            b.set_verify(16, 0.01)
        b.run(160, sync_every=20)
        part = b.status_array()
        assert (part["kind"] == 3).any() and (part["force_calls"][part["done"] == 0] == 260).all()
        b.run(400, sync_every=20)
        out.append((part, b.status_array(), b.positions()))
    for k in out[0][0].dtype.names:
        assert np.array_equal(out[0][0][k], out[1][0][k], equal_nan=True), k
        assert np.array_equal(out[0][1][k], out[1][1][k], equal_nan=True), k
    assert (out[0][1]["verified"] == 1).any()
    for p, q in zip(out[0][2], out[1][2]):
        assert np.array_equal(p, q)
