"""The plain force call at the edges of its kernel variants: a wavefront per
atom below 16,384 atoms and 8 lanes from there, pair tables with n = 9, m = 6
throughout (straight products) and with other exponents, one and two atoms,
with and without stress and minimum images; and transfers on both sides of the
pinned-buffer limit.  Each against the one-lane kernels of a batch on the same
cell: the same pair terms summed in another order, 1e-12 of the largest force
(FP32 pair terms enter FP64 sums unrounded)."""
import numpy as np
import pytest

from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
CU = W.SC_CU
ONE = [("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])]
GENERAL = [("Cu", "Cu", 0.0124, 3.61, 9.0, 6.0, 39.4), ("Ni", "Ni", 0.0158, 3.52, 10.0, 8.0, 34.4),
           ("Cu", "Ni", 0.0140, 3.57, 9.5, 7.0, 36.8)]
POTS = dict(one=ONE, alloy=W.ALLOY_POTS, general=GENERAL)


def _check(L, f, c, stress):
    b = L.Batch(f, [c])
    b.set_variant(1, 1)
    e = b.forces()[0]
    ref = b.download()[1][0]
    got = f.calculate_forces(c.pos, c.types, c.lat, stress=stress)
    scale = max(1.0, np.abs(ref).max())
    assert np.abs(got["force"] - ref).max() < 1e-12 * scale
    assert abs(got["energy"]["total"] - e["total"]) <= 1e-12 * max(1.0, abs(e["total"]))
    again = f.calculate_forces(c.pos, c.types, c.lat, stress=stress)
    assert np.array_equal(again["force"], got["force"]) and again["energy"] == got["energy"]


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("kind,shape,vac,noimage", [
    ("one", (4, 4, 4), 1, False), ("one", (4, 4, 4), 1, True), ("one", (16, 16, 16), 1, False),
    ("one", (16, 16, 16), 0, False), ("alloy", (5, 5, 6), 3, False), ("alloy", (16, 16, 17), 5, False),
    ("general", (5, 6, 5), 2, False), ("general", (5, 6, 5), 2, True)])
def test_variants_agree(kind, shape, vac, noimage, bits):
    from akmc_amd import lib as L
    c = W.sc_cell(*shape, n_vac=vac, jitter=0.05, seed=3, two_species=kind != "one", a=3.65)
    f = L.Field(L.sc_potentials_text(POTS[kind], 2 * CU["a"], species=["Cu"] if kind == "one" else ["Cu", "Ni"],
                                     noimage=noimage))
    f.set_precision(bits)
    for stress in (False, True):
        if kind == "alloy" and bits == 32 and stress:
            continue  # the stress kernels take the general powers: another rounding of each FP32 term
        _check(L, f, c, stress)


@pytest.mark.parametrize("n", [1, 2])
def test_one_and_two_atoms(n):
    from akmc_amd import lib as L
    lat = np.diag([16.0] * 3).reshape(9)
    pos = np.array([[1.0, 3.4], [2.0, 2.1], [3.0, 3.0]])[:, :n].copy()
    c = W.Cell(pos, np.zeros(n, np.int32), lat, ["Cu"])
    f = L.Field(L.sc_potentials_text(ONE, 2 * CU["a"]))
    f.set_list_density(0.01)
    _check(L, f, c, False)
