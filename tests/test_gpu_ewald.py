"""The reciprocal Ewald kernels at the edges of their tiles, in batches of
cells of different sizes: 1 to 4 atoms in a workgroup's last group of four,
fewer atoms than a tile of k has summing threads, k counts below one 32-k tile
(17 at g = 2) and past one and just short of two rounds of the force kernel's
256 threads (276 and 501), and tables too long for LDS (67 entries).  FP64 pair terms against the oracle: forces 1e-8 eV/A, energies
1e-10 eV per atom, as its other FP64 comparisons."""
import numpy as np
import pytest

from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
POTS = [k + W.ROCKSALT_BUCK[k] for k in (("M", "X"), ("X", "X"), ("M", "M"))]


def _cut(c, n):
    """the cell's first n ions"""
    return W.Cell(np.ascontiguousarray(c.pos[:, :n]), c.types[:n].copy(), c.lat, c.species, charges=c.charges[:n].copy())


@pytest.mark.parametrize("g", [2, 5, 6, 66])
def test_reciprocal_sums(oracle, g):
    from akmc_amd import lib as L
    eta = 0.35
    full = W.rocksalt_cell(1, 1, 14, seed=2, schottky=False) if g == 66 else W.rocksalt_cell(2, 2, 2, seed=2, schottky=False)
    cells = [_cut(full, n) for n in ([112, 109] if g == 66 else [61, 64, 1, 63, 62])]
    f = L.Field(L.buck_potentials_text(["M", "X"], [2.0, -2.0], POTS, 10.0, noimage=True))
    f.set_precision(64)
    f.set_list_density(0.2)
    f.set_ewald(eta, g)
    b = L.Batch(f, cells)
    e = b.forces()
    F = b.download()[1]
    for w, c in enumerate(cells):
        of = oracle.ion_field(["M", "X"], POTS, rc=10.0, ewald=oracle.Ewald(c.lat, eta, gcell=g), min_image=False,
                              lat=c.lat)
        ref = oracle.ion_forces(of, c.pos, c.types, c.charges, c.lat)
        assert np.abs(F[w] - ref["force"]).max() < 1e-8
        assert abs(e[w]["rcp"] - ref["e_rcp"]) < 1e-10 * c.n
        assert abs(e[w]["real"] - ref["e_real"]) < 1e-10 * c.n
