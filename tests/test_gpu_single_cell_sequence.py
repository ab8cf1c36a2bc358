"""Plain force calls on cells of changing size through one field: the pinned
transfer buffer passes from cell to cell, grows, and stays out of the calls
past its limit (4 MiB, about 75,000 atoms).  Each call gives the bits that a
field of its own gives."""
import numpy as np
import pytest

from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
CU = W.SC_CU


def test_cells_of_changing_size():
    from akmc_amd import lib as L

    def field():
        return L.Field(L.sc_potentials_text([("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])], 2 * CU["a"]))

    shapes = [(4, 4, 4), (5, 5, 5), (4, 4, 4), (27, 27, 27), (6, 4, 4), (5, 5, 5), (4, 4, 5)]
    f = field()
    for k, shape in enumerate(shapes):
        c = W.sc_cell(*shape, n_vac=1, jitter=0.02, seed=k)
        for stress in (False, True):
            got = f.calculate_forces(c.pos.copy(), c.types, c.lat, stress=stress)
            ref = field().calculate_forces(c.pos.copy(), c.types, c.lat, stress=stress)
            assert np.array_equal(got["force"], ref["force"]) and got["energy"] == ref["energy"]
        assert f.calculate_energy(c.pos.copy(), c.types, c.lat) == field().calculate_energy(c.pos.copy(), c.types, c.lat)
