"""Calls that change a running search's inputs between chunks of micro-steps:
the search goes on with the new inputs, whichever kernels advance it.

The end of a FIRE relax is compared with a force call of the whole cell at
its positions: FP64, the same terms in another order, 1e-11.
"""
import numpy as np
import pytest

from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
CU = W.SC_CU
ONE = [("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])]


def _field():
    from akmc_amd import lib as L
    f = L.Field(L.sc_potentials_text(ONE, 2 * CU["a"]))
    f.set_precision(64)
    return L, f


def _frozen(c, nfree):
    frozen = np.ones(c.n, np.int32)
    frozen[np.argsort(W.site_distances(c, c.vacancies[0]), kind="stable")[:nfree]] = 0
    return frozen


def _check(f, c, pos, force, energy, free):
    ref = f.calculate_forces(pos.copy(), c.types, c.lat, stress=False)
    assert np.abs(force - ref["force"])[:, free].max() < 1e-11
    assert abs(energy - ref["energy"]["total"]) < 1e-11 * abs(ref["energy"]["total"])


def test_new_positions_under_a_running_search():
    L, f = _field()
    cells = [W.sc_cell(4, 4, 5, n_vac=1, jitter=0.02, seed=s) for s in (1, 2)]
    frozen = [_frozen(c, 60) for c in cells]
    b = L.Batch(f, cells)
    b.set_frozen(frozen)
    b.start_relax(L.relax_defaults(maxIter=40, maxTimeStep=0.003, initTimeStep=0.002))
    b.run(10, sync_every=5)
    calls = [s["force_calls"] for s in b.status()]
    assert all(k == calls[0] for k in calls) and 0 < calls[0] <= 10
    moved = [W.sc_cell(4, 4, 5, n_vac=1, jitter=0.03, seed=s) for s in (3, 4)]
    moved = [W.Cell(m.pos, c.types, c.lat) for m, c in zip(moved, cells)]
    b.upload(moved)
    b.run(200, sync_every=13)
    st, pos, frc = b.status(), b.positions(), b.download()[1]
    for w, c in enumerate(moved):
        assert st[w]["done"] == 1 and st[w]["force_calls"] > calls[w]
        fixed = frozen[w] == 1
        assert np.array_equal(pos[w][:, fixed], c.pos[:, fixed])
        _check(f, c, pos[w], frc[w], st[w]["energy"], ~fixed)


@pytest.mark.parametrize("nfree", [20, 64, 300])
def test_new_frozen_mask_under_a_running_search(nfree):
    """Fewer free atoms, a few more, and more than a resident walker takes,
    for one of two walkers; the other keeps its mask."""
    L, f = _field()
    cells = [W.sc_cell(4, 4, 6, n_vac=1, jitter=0.02, seed=s) for s in (1, 2)]
    frozen = [_frozen(c, 60) for c in cells]
    b = L.Batch(f, cells)
    b.set_frozen(frozen)
    b.start_relax(L.relax_defaults(maxIter=40, maxTimeStep=0.003, initTimeStep=0.002))
    b.run(10, sync_every=5)
    part = b.positions()
    assert (b.zone()[2] & 16).all()
    frozen[0] = _frozen(cells[0], nfree)
    b.set_frozen(frozen)
    b.run(300, sync_every=13)
    flags = b.zone()[2]
    assert not flags[0] & 16 and flags[1] & 16
    st, pos, frc = b.status(), b.positions(), b.download()[1]
    for w, c in enumerate(cells):
        assert st[w]["done"] == 1
        fixed = frozen[w] == 1
        assert np.array_equal(pos[w][:, fixed], part[w][:, fixed])
        assert np.abs(pos[w] - part[w])[:, ~fixed].max() > 1e-4
        _check(f, c, pos[w], frc[w], st[w]["energy"], ~fixed)


def test_refused_start_leaves_masks_alone():
    """A start refused for one walker's zero mode, with masks that would let
    the walkers run resident, changes no walker's mask: the relax after it
    moves the atoms that were free before."""
    L, f = _field()
    cells = [W.sc_cell(5, 5, 5, n_vac=1, jitter=0.02, seed=s) for s in (1, 2)]
    frozen = [_frozen(c, 300) for c in cells]
    b = L.Batch(f, cells)
    b.set_frozen(frozen)
    modes = [np.ones((3, cells[0].n)), np.zeros((3, cells[1].n))]
    with pytest.raises(L.AkmcError, match="zero start mode"):
        b.start_dimer(modes, frozen_per_walker=[_frozen(c, 60) for c in cells])
    with pytest.raises(L.AkmcError, match="relax method"):
        b.start_relax_at(None, frozen=np.concatenate([_frozen(c, 60) for c in cells]),
                         params=L.relax_defaults(method=7))
    b.start_relax(L.relax_defaults(maxIter=20, maxTimeStep=0.003, initTimeStep=0.002))
    b.run(300, sync_every=13)
    st, pos, frc = b.status(), b.positions(), b.download()[1]
    for w, c in enumerate(cells):
        assert st[w]["done"] == 1
        moved = np.abs(pos[w] - c.pos).max(0) > 0
        assert np.array_equal(moved, frozen[w] == 0)
        _check(f, c, pos[w], frc[w], st[w]["energy"], frozen[w] == 0)


def test_variants_are_timed_on_the_pair_kernels():
    """autotune_search under resident searches times the pair kernels'
    evaluation of all the walkers' atoms (the forces it leaves are those of a
    force call at the probes, frozen atoms included) and changes no search."""
    from akmc_amd import lib as L
    f = L.Field(L.sc_potentials_text(ONE, 2 * CU["a"]))
    cells = [W.sc_cell(4, 4, 6, n_vac=1, jitter=0.02, seed=s) for s in (1, 2)]
    frozen = [_frozen(c, 60) for c in cells]
    ends = []
    for tune in (True, False):
        b = L.Batch(f, cells)
        b.set_frozen(frozen)
        b.start_relax(L.relax_defaults(maxIter=60, maxTimeStep=0.003, initTimeStep=0.002))
        b.run(30, sync_every=10)
        flags = b.zone()[2]
        assert (flags & 16).all()
        if tune:
            best, ms = b.autotune_search(2)
            assert np.array_equal(b.zone()[2], flags) and all(v[0] > 0 and v[1] > 0 for v in ms.values())
            pos, frc = b.download()
            for w, c in enumerate(cells):
                ref = f.calculate_forces(pos[w].copy(), c.types, c.lat, stress=False)
                assert np.abs(frc[w] - ref["force"]).max() < 2e-5
        b.run(300, sync_every=10)
        ends.append((b.positions(), b.status_array()))
    assert (ends[0][1]["done"] == 1).all()
    for k in ends[0][1].dtype.names:
        assert np.array_equal(ends[0][1][k], ends[1][1][k], equal_nan=True), k
    for p, q in zip(ends[0][0], ends[1][0]):
        assert np.array_equal(p, q)
