"""Which walkers the resident kernel takes, and its evaluation over the range:
more than 128 free atoms (the upper bits of the mask words), free-atom lists
too long for LDS, list builds in more than one strip of hit words, up to 256
free atoms.  zone()'s flag 16 tells that the walker stayed resident to the
end; the energy and the free atoms' forces there are those of a force call of
the whole cell (FP64: the same terms in another order, 1e-11; FP32: 2e-5 eV/A
and 1e-6 eV per atom, the budget of the field tests).
"""
import numpy as np
import pytest

from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
CU = W.SC_CU
ONE = [("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])]


def _relax(cells, frozen, bits, run=400, sync=13):
    from akmc_amd import lib as L
    f = L.Field(L.sc_potentials_text(ONE, 2 * CU["a"]))
    f.set_precision(bits)
    b = L.Batch(f, cells)
    b.set_frozen(frozen)
    b.start_relax(L.relax_defaults(maxIter=25, maxTimeStep=0.003, initTimeStep=0.002))
    b.run(run, sync_every=sync)
    return f, b


def _nearest(c, n, site=None):
    frozen = np.ones(c.n, np.int32)
    frozen[np.argsort(W.site_distances(c, c.vacancies[0] if site is None else site), kind="stable")[:n]] = 0
    return frozen


def _check(f, b, cells, frozen, bits):
    st, pos, frc = b.status(), b.positions(), b.download()[1]
    for w, c in enumerate(cells):
        ref = f.calculate_forces(pos[w].copy(), c.types, c.lat, stress=False)
        assert st[w]["done"] == 1 and st[w]["force_calls"] >= 2
        df = np.abs(frc[w] - ref["force"])[:, frozen[w] == 0].max()
        de = abs(st[w]["energy"] - ref["energy"]["total"])
        print(f"{c.n} atoms, {(frozen[w] == 0).sum()} free, fp{bits}: max|dF| {df:.2e}, |dE| {de:.2e}", flush=True)
        assert df < (1e-11 if bits == 64 else 2e-5)
        assert de < (1e-11 * abs(ref["energy"]["total"]) if bits == 64 else 1e-6 * c.n)


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("shape,nfree", [((8, 8, 8), 129), ((10, 10, 10), 200), ((10, 10, 10), 212),
                                         ((10, 10, 10), 213), ((8, 8, 8), 256), ((10, 10, 10), 256)])
def test_compact_region_is_resident(shape, nfree, bits):
    c = W.sc_cell(*shape, n_vac=1, jitter=0.02, seed=5)
    frozen = _nearest(c, nfree)
    f, b = _relax([c], [frozen], bits)
    assert b.zone()[2][0] & 16
    _check(f, b, [c], [frozen], bits)


def test_one_free_atom_more_takes_the_chain():
    c = W.sc_cell(8, 8, 8, n_vac=1, jitter=0.02, seed=5)
    frozen = _nearest(c, 257)
    f, b = _relax([c], [frozen], 64)
    assert not b.zone()[2][0] & 16
    _check(f, b, [c], [frozen], 64)


def test_two_separated_clusters_are_resident():
    c = W.sc_cell(10, 10, 10, n_vac=1, jitter=0.02, seed=6)
    frozen = _nearest(c, 60)
    other = np.asarray(c.vacancies[0]) + 5 * CU["a"] * np.array([1.0, 1.0, 1.0])
    frozen &= _nearest(c, 60, other)
    assert (frozen == 0).sum() == 120
    f, b = _relax([c], [frozen], 64)
    assert b.zone()[2][0] & 16
    _check(f, b, [c], [frozen], 64)


def _scattered(c, n, seed):
    frozen = np.ones(c.n, np.int32)
    frozen[np.random.default_rng(seed).choice(c.n, n, replace=False)] = 0
    return frozen


def test_a_walker_that_does_not_fit_leaves_the_others_alone():
    """A small search beside one whose 200 scattered free atoms reach more
    than 2048 atoms, and beside a cell past 16383 atoms: the same bits as
    alone, at the first start and after a restart; only the others are on the
    chain, and they make a force call a step from their first step on."""
    from akmc_amd import lib as L
    small = W.sc_cell(4, 4, 5, n_vac=1, jitter=0.02, seed=1)
    wide = W.sc_cell(9, 9, 9, n_vac=1, jitter=0.02, seed=2)
    huge = W.sc_cell(16, 16, 17, n_vac=1, jitter=0.02, seed=3)
    cells = [small, wide, huge]
    frozen = [_nearest(small, 60), _scattered(wide, 200, 1), _nearest(huge, 60)]
    f, alone = _relax([small], [frozen[0]], 32, run=9, sync=9)
    f, b = _relax(cells, frozen, 32, run=9, sync=9)
    for again in range(2):
        st, one = b.status(), alone.status()
        assert [int(v) & 16 for v in b.zone()[2]] == [16, 0, 0] and alone.zone()[2][0] & 16
        assert [s["force_calls"] for s in st] == [9, 9, 9]
        for bb in (b, alone):
            bb.run(400, sync_every=9)
        st, one = b.status(), alone.status()
        assert st[0] == one[0] and st[0]["done"] == 1
        assert np.array_equal(b.positions()[0], alone.positions()[0])
        if again == 0:
            _check(f, b, cells, frozen, 32)
            for bb in (b, alone):
                bb.start_relax(L.relax_defaults(maxIter=25, maxTimeStep=0.004, initTimeStep=0.003))
                bb.run(9, sync_every=9)


def _zone(c, pos, frozen, reach):
    free = np.nonzero(frozen == 0)[0]
    inz = frozen == 0
    for i in free:
        inz |= W.site_distances(W.Cell(pos, c.types, c.lat), pos[:, i]) <= reach
    return int(inz.sum())


def _outgrowing(seed):
    """16 scattered free atoms of a perfect lattice, displaced: (cell, mask,
    zone at the start, zone when the farthest one has come back by half the
    skin, skin)"""
    c = W.sc_cell(10, 10, 10, n_vac=1, jitter=0.0, seed=4)
    skin = 1.2
    frozen = _scattered(c, 16, seed)
    disp = np.where(frozen == 0, np.random.default_rng(seed).uniform(-0.6, 0.6, (3, c.n)), 0.0)
    t = 1 - skin / 2 / np.sqrt((disp ** 2).sum(0)).max()
    reach = 2 * CU["a"] + skin / 2
    return (W.Cell(c.pos + disp, c.types, c.lat, vacancies=c.vacancies), frozen,
            _zone(c, c.pos + disp, frozen, reach + 0.01), _zone(c, c.pos + t * disp, frozen, reach - 0.01), skin)


def test_a_zone_that_outgrows_the_kernel_goes_on_in_the_chain():
    """16 scattered free atoms whose zone has at most 2048 atoms at the start
    of a relax and more when they have come back."""
    cell, frozen, z0, z1, skin = _outgrowing(20)
    assert z0 <= 2044 and z1 >= 2060
    from akmc_amd import lib as L
    f = L.Field(L.sc_potentials_text(ONE, 2 * CU["a"]))
    f.set_precision(64)
    f.set_skin(skin)
    b = L.Batch(f, [cell])
    b.set_frozen([frozen])
    b.start_relax(L.relax_defaults(maxIter=400, maxTimeStep=0.004, initTimeStep=0.003))
    assert b.zone()[2][0] & 16
    b.run(3000, sync_every=10)
    assert not b.zone()[2][0] & 16
    _check(f, b, [cell], [frozen], 64)


def test_starts_behind_a_chunk_in_flight():
    """Two walkers started while a chunk runs, one that fits the resident
    kernel and one that does not: both take a step with every micro-step of
    the next chunk, and end as they do when started before it."""
    from akmc_amd import lib as L
    cells = [W.sc_cell(4, 4, 5, n_vac=1, jitter=0.02, seed=1), W.sc_cell(5, 4, 5, n_vac=1, jitter=0.02, seed=4),
             W.sc_cell(9, 9, 9, n_vac=1, jitter=0.02, seed=2)]
    frozen = [_nearest(cells[0], 60), _nearest(cells[1], 70), _scattered(cells[2], 200, 1)]
    f = L.Field(L.sc_potentials_text(ONE, 2 * CU["a"]))
    modes, x0 = [], []
    for w, c in enumerate(cells):
        disp, mode = W.local_displacement(c, W.neighbours_of_site(c, c.vacancies[0], 12), 0.1, w)
        modes.append(mode)
        x0.append(c.pos + disp)
    modes[2] = np.random.default_rng(1).standard_normal((3, cells[2].n))  # its free atoms are everywhere
    ends = []
    for behind in (True, False):
        b = L.Batch(f, cells)
        kw = dict(x0_per_walker=x0, frozen_per_walker=frozen)
        b.start_dimer(modes, walkers=[0], **kw)
        if behind:
            b.run_async(20)
            b.start_dimer(modes, walkers=[1, 2], **kw)
            b.run_wait()
        else:
            b.run(20, sync_every=20)
            b.start_dimer(modes, walkers=[1, 2], **kw)
        assert [int(v) & 16 for v in b.zone()[2]] == [16, 16, 0]
        for _ in range(2):
            b.run_next(15) if behind else b.run_async(15)
            b.run_wait()
        assert [s["force_calls"] for s in b.status()] == [50, 30, 30]
        ends.append(b.positions())
    for p, q in zip(*ends):
        assert np.array_equal(p, q)
