"""Device descriptors and the fused network kernels at the edges of their
ranges: queries that repeat atoms in any order across walkers of different
sizes, a single query, atoms with few neighbours; network batches of one row,
around the 64-row tile and past the gradient kernel's 256 workgroups.

Descriptors are FP32 sums of up to a few hundred terms against the FP64
oracle: 1e-4 relative (values below 1e-3: absolute), the budget of the
descriptor test.  The network rounds operands to BF16 (2^-9 relative) over
K <= 128: 3e-2 norm-wise, the budget of the network test; a gradient of one
row has a single term per weight, of the same budget.
"""
import numpy as np
import pytest

from akmc_amd import workloads as W
from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu
CU = W.SC_CU


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("nq", [1, 63, 700])
def test_repeated_atoms_match_oracle(nq):
    from akmc_amd import learn as LN
    from akmc_amd import lib as L
    cells = [W.sc_cell(4, 4, 4, 1, 0.05, 3), W.sc_cell(5, 4, 6, 2, 0.05, 4)]
    # a sparse walker: most atoms removed, so some have no neighbour inside 5 A
    c = W.sc_cell(6, 6, 6, 1, 0.05, 5)
    keep = np.sort(np.random.default_rng(2).choice(c.n, 60, replace=False))
    cells.append(W.Cell(np.ascontiguousarray(c.pos[:, keep]), c.types[keep], c.lat, c.species, vacancies=c.vacancies))
    f = L.Field(L.sc_potentials_text([("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])], 2 * CU["a"]))
    f.set_list_density(4 / CU["a"] ** 3)
    b = L.Batch(f, cells)
    b.forces()
    rng = np.random.default_rng(nq)
    w = rng.integers(0, 3, nq)
    a = np.array([rng.integers(0, min(cells[k].n, 20)) for k in w])  # many repeats
    vac = np.stack([cells[k].vacancies[0] + rng.normal(0, 1.0, 3) for k in w])
    mov = np.stack([cells[k].pos[:, int(rng.integers(0, cells[k].n))] for k in w])
    X = LN.batch_descriptors(b, b.offsets[w] + a, vac, mov)
    assert X.shape == (nq, 48) and np.isfinite(X).all()
    for q in range(0, nq, max(1, nq // 12)):
        k = w[q]
        R = MO.descriptors(cells[k].pos, cells[k].lat, [int(a[q])], vac[q], mov[q])[0]
        err = np.abs(X[q] - R) / np.maximum(np.abs(R), 1e-3)
        assert err.max() < 1e-4, (q, int(err.argmax()), err.max())
    for k in range(3):
        for i in np.unique(a[w == k]):
            rows = X[(w == k) & (a == i)]
            assert np.array_equal(rows[:, :16], np.tile(rows[:1, :16], (len(rows), 1)))
            assert np.array_equal(rows[:, 32:], np.tile(rows[:1, 32:], (len(rows), 1)))


@pytest.mark.parametrize("M", [1, 16, 63, 64, 65, 4097, 16384 + 129])
def test_network_tile_edges_match_oracle(M):
    from akmc_amd import learn as LN
    rng = np.random.default_rng(M)
    p = MO.init_params(7)
    for k in ("b1", "b2"):
        p[k] = rng.normal(0, 0.1, 128)
    p["b3"] = rng.normal(0, 0.1, 3)
    X, T = rng.normal(size=(M, 48)), rng.normal(size=(M, 3))
    net = LN.MLP(max_rows=20000)
    net.params = LN.pack(p)
    Yr, _ = MO.forward(p, X)
    assert _rel(net.forward(X), Yr) < 3e-2
    loss, g = net.loss_grad(X, T)
    lr, gr = MO.loss_and_grad(p, X, T)
    assert abs(loss - lr) < 3e-2 * lr
    gd = LN.unpack(g)
    for k in ("W1", "b1", "W2", "b2", "W3", "b3"):
        assert _rel(gd[k], gr[k]) < 3e-2, k
