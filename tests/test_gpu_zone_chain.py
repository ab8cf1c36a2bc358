"""Searches with the resident kernel off: active zones against full
evaluations by the same pair kernels, bit for bit, and the resident kernel
against them.

The resident kernel adds the same terms in another order, so the first
evaluation of a search agrees with a full one to the rounding of FP64 sums
of a few hundred terms (forces up to a few eV/A: 1e-11; energies of a few
thousand eV: 1e-12 of them), in both precisions.
"""
import numpy as np
import pytest

from test_gpu_zone import CU, _cells, _starts, _text  # noqa: F401
from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
POTS = {"alloy": W.ALLOY_POTS,
        "general": [("Cu", "Cu", 0.0124, 3.61, 9.0, 6.0, 39.4), ("Ni", "Ni", 0.0158, 3.52, 10.0, 8.0, 34.4),
                    ("Cu", "Ni", 0.0140, 3.57, 9.5, 7.0, 36.8)]}


@pytest.fixture(scope="module")
def lib():
    from akmc_amd import lib as L
    L.load()
    return L


def _run(lib, cells, zone):
    """relax, then dimer + FP64 verification + basin 2 on every walker"""
    f = lib.Field(_text(lib))
    b = lib.Batch(f, cells)
    b.set_resident(False)
    b.set_search_zone(zone)
    b.set_frozen([np.zeros(c.n, np.int32) for c in cells])
    b.start_relax(lib.relax_defaults())
    b.run(20000, sync_every=50)
    frozen, modes, x0 = _starts(cells, b.positions(), 11)
    b.set_basins()
    b.set_basin2(lib.basin2_defaults())
    b.set_verify(16, 0.01)
    b.start_dimer(modes, params=lib.dimer_defaults(maxParIter=400), x0_per_walker=x0, frozen_per_walker=frozen)
    assert not (b.zone()[2] & 16).any()
    b.run(40000, sync_every=25)
    return dict(status=b.status_array(), pos=b.positions(), saddles=b.walkers_saddles(list(range(len(cells)))),
                forces=b.download()[1], frozen=frozen)


def test_zones_equal_full_evaluations_bitwise(lib):
    cells = _cells()
    on, off = _run(lib, cells, True), _run(lib, cells, False)
    for k in on["status"].dtype.names:
        assert np.array_equal(on["status"][k], off["status"][k], equal_nan=True), k
    assert (on["status"]["done"] == 1).all() and (on["status"]["verified"] == 1).any()
    stale = 0
    for w in range(len(cells)):
        assert np.array_equal(on["pos"][w], off["pos"][w])
        assert np.array_equal(on["saddles"][w], off["saddles"][w])
        free = on["frozen"][w] == 0
        assert np.array_equal(on["forces"][w][:, free], off["forces"][w][:, free])
        stale += np.abs(on["forces"][w][:, ~free] - off["forces"][w][:, ~free]).max() > 1e-6
    assert stale >= len(cells) // 2


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("kind", ["one", "alloy", "general"])
def test_resident_evaluation_equals_the_pair_kernels(lib, kind, bits):
    if kind == "one":
        f = lib.Field(_text(lib))
        cells = _cells()
    else:
        f = lib.Field(lib.sc_potentials_text(POTS[kind], 2 * CU["a"], species=["Cu", "Ni"]))
        cells = [W.sc_cell(n, 5, 6, n_vac=1, jitter=0.02, seed=n, two_species=True, a=3.65) for n in (5, 6, 7)]
    f.set_precision(bits)
    out = []
    for resident in (True, False):
        b = lib.Batch(f, cells)
        b.set_resident(resident)
        frozen, modes, x0 = _starts(cells, [c.pos for c in cells], 11)
        b.start_dimer(modes, x0_per_walker=x0, frozen_per_walker=frozen)
        assert (((b.zone()[2] & 16) != 0) == resident).all()
        b.run(1, sync_every=1)
        out.append((b.status_array()["energy"].copy(), b.download()[1]))
    for w, c in enumerate(cells):
        free = frozen[w] == 0
        d = np.abs(out[0][1][w] - out[1][1][w])
        de = abs(out[0][0][w] / out[1][0][w] - 1)
        print(f"{kind} fp{bits} {c.n} atoms: max|dF| {d[:, free].max():.1e}, dE/E {de:.1e}", flush=True)
        assert d[:, free].max() < 1e-11 and de < 1e-12
        assert np.array_equal(out[0][1][w][:, ~free], out[1][1][w][:, ~free])
