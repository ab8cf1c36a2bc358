"""Resident searches (search_resident.hip) at the edges of their ranges: one
free atom, the most free atoms a resident walker takes and one more (the
chain), a scattered free set that reaches more atoms than one holds (the
chain), cells smaller and larger than the zone, and the three
kinds of pair table (one species; n = 9, m = 6 throughout; any exponents),
in both precisions.

Every case relaxes with frozen atoms for a few FIRE iterations and compares
the energy and the free atoms' forces at the end with a force call of the
whole cell at those positions.  FP64: the same terms in another order, sums
of a few hundred terms of order 1: 1e-11.  FP32: each pair term within a few
2^-24 of its value, terms up to a few eV/A: 2e-5 eV/A on a force (the budget
of the field tests) and 1e-6 eV per atom.
"""
import numpy as np
import pytest

from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
CU = W.SC_CU
ONE = [("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])]
GENERAL = [("Cu", "Cu", 0.0124, 3.61, 9.0, 6.0, 39.4), ("Ni", "Ni", 0.0158, 3.52, 10.0, 8.0, 34.4),
           ("Cu", "Ni", 0.0140, 3.57, 9.5, 7.0, 36.8)]


def _case(kind, shape, seed):
    if kind == "one":
        return W.sc_cell(*shape, n_vac=1, jitter=0.02, seed=seed), ONE, ["Cu"]
    c = W.sc_cell(*shape, n_vac=1, jitter=0.02, seed=seed, two_species=True, a=3.65)
    return c, (W.ALLOY_POTS if kind == "alloy" else GENERAL), ["Cu", "Ni"]


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("kind,shape,nfree,scattered", [
    ("one", (4, 4, 4), 1, False),
    ("one", (4, 4, 7), 78, False),
    ("one", (8, 8, 8), 256, False),
    ("one", (8, 8, 8), 257, False),
    ("one", (9, 9, 9), 200, True),
    ("alloy", (5, 6, 7), 65, False),
    ("general", (6, 6, 6), 64, False),
])
def test_resident_evaluation_equals_force_call(kind, shape, nfree, scattered, bits):
    from akmc_amd import lib as L
    c, pots, species = _case(kind, shape, 5)
    f = L.Field(L.sc_potentials_text(pots, 2 * CU["a"], species=species))
    f.set_precision(bits)
    if scattered:
        free = np.random.default_rng(1).choice(c.n, nfree, replace=False)
    else:
        free = np.argsort(W.site_distances(c, c.vacancies[0]), kind="stable")[:nfree]
    frozen = np.ones(c.n, np.int32)
    frozen[free] = 0
    b = L.Batch(f, [c, c])
    b.set_frozen([frozen, frozen])
    b.start_relax(L.relax_defaults(maxIter=30, maxTimeStep=0.003, initTimeStep=0.002))
    b.run(400, sync_every=13)
    assert (((b.zone()[2] & 16) != 0) == (nfree <= 256 and not scattered)).all()  # which path it was
    st = b.status()
    pos = b.positions()
    frc = b.download()[1]
    assert all(s["done"] == 1 for s in st)
    assert st[0]["force_calls"] == st[1]["force_calls"] >= 2
    assert np.array_equal(pos[0], pos[1]) and st[0]["energy"] == st[1]["energy"]
    assert np.array_equal(pos[0][:, frozen == 1], c.pos[:, frozen == 1])
    assert np.abs(pos[0] - c.pos).max() > 1e-3
    ref = f.calculate_forces(pos[0].copy(), c.types, c.lat, stress=False)
    df = np.abs(frc[0] - ref["force"])[:, frozen == 0].max()
    de = abs(st[0]["energy"] - ref["energy"]["total"])
    print(f"{kind} {shape} {nfree} free, fp{bits}: {st[0]['force_calls']} calls, max|dF| {df:.2e}, |dE| {de:.2e}", flush=True)
    assert df < (1e-11 if bits == 64 else 2e-5)
    assert de < (1e-11 * abs(ref["energy"]["total"]) if bits == 64 else 1e-6 * c.n)
