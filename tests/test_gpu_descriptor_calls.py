"""Descriptors need lists and positions alone: they are given for a batch
whose force call failed on its embedding table, as for any other."""
import numpy as np
import pytest

import eam_fixtures as FX
from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
CU = W.SC_CU


def test_descriptors_after_a_failed_embedding(tmp_path):
    from akmc_amd import learn as LN
    from akmc_amd import lib as L
    c = W.plain_sc_workload(seed=1)
    rc = 2 * CU["a"]
    short = FX.sc_setfl(tmp_path / "short.eam", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"], rc, rho_max=10.0)
    site = c.vacancies[0]
    mover = int(np.argmin(W.site_distances(c, site)))
    atoms = np.argsort(W.site_distances(c, site))[:40]
    query = (atoms, np.tile(site, (40, 1)), np.tile(c.pos[:, mover], (40, 1)))
    b = L.Batch(L.Field(L.eam_potentials_text([("Cu", "Cu", str(short))], rc)), [c])
    with pytest.raises(L.AkmcError, match="out of bounds"):
        b.forces()
    got = LN.batch_descriptors(b, *query)
    b = L.Batch(L.Field(L.sc_potentials_text([("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])], rc)), [c])
    b.forces()
    ref = LN.batch_descriptors(b, *query)
    assert np.abs(ref).max() > 0.1 and np.abs(got - ref).max() < 1e-4
