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


def test_two_separated_clusters_are_resident():
    c = W.sc_cell(10, 10, 10, n_vac=1, jitter=0.02, seed=6)
    frozen = _nearest(c, 60)
    other = np.asarray(c.vacancies[0]) + 5 * CU["a"] * np.array([1.0, 1.0, 1.0])
    frozen &= _nearest(c, 60, other)
    assert (frozen == 0).sum() == 120
    f, b = _relax([c], [frozen], 64)
    assert b.zone()[2][0] & 16
    _check(f, b, [c], [frozen], 64)
