"""List builds and the plain FIRE step at the edges of their kernels.

A cell past 8,192 atoms is binned in segments of 1,024 atoms, a smaller one by
one workgroup; explicit-image lists take 27 images as masks where one shell
per axis is enough and loop over the shells otherwise.  Both are checked with
periodic copies: the same infinite crystal, so the same forces.  FP64 pair
terms; a coordinate of up to 200 A rounds at 2.8e-14 A, times a stiffness of
some 20 eV/A^2 and 150 pairs: 1e-10 eV/A."""
import numpy as np
import pytest

from akmc_amd import workloads as W

pytestmark = pytest.mark.gpu
CU = W.SC_CU
ONE = [("Cu", "Cu", CU["eps"], CU["a"], CU["n"], CU["m"], CU["c"])]
RC = 7.0  # no multiple of a lattice constant: an atom's own copies are never at the cutoff itself


def _forces(c, noimage=False):
    from akmc_amd import lib as L
    f = L.Field(L.sc_potentials_text(ONE, RC, species=["Cu"], noimage=noimage))
    f.set_precision(64)
    b = L.Batch(f, [c])
    e = b.forces()[0]
    return e["total"], b.download()[1][0]


def _copies(c, reps):
    """the cell repeated reps times along each axis, copy after copy"""
    d = np.asarray(c.lat).reshape(3, 3).diagonal()
    pos = [c.pos + (np.array([i, j, k]) * d)[:, None]
           for i in range(reps[0]) for j in range(reps[1]) for k in range(reps[2])]
    return W.Cell(np.ascontiguousarray(np.concatenate(pos, 1)), np.tile(c.types, len(pos)),
                  np.diag(d * np.array(reps)).reshape(9), c.species)


def _same(c, big, reps, **kw):
    e, f = _forces(c, **kw)
    eb, fb = _forces(big, **{**kw, "noimage": False})
    m = int(np.prod(reps))
    assert np.abs(fb - np.tile(f, (1, m))).max() < 1e-10
    assert abs(eb - m * e) < 1e-10 * abs(eb)


# atoms of the copied cell: the most that one workgroup bins (8,192), and cells
# whose last segment is full (16,384), nearly full (9,212) or shorter
@pytest.mark.parametrize("shape,vac,reps", [((8, 8, 8), 0, (2, 2, 1)), ((8, 8, 8), 0, (2, 2, 2)),
                                            ((6, 6, 22), 0, (1, 1, 3)), ((8, 8, 11), 1, (2, 2, 1)),
                                            ((8, 8, 9), 1, (2, 2, 1))])
def test_segmented_binning(shape, vac, reps):
    c = W.sc_cell(*shape, n_vac=vac, jitter=0.05, seed=5)
    _same(c, _copies(c, reps), reps)


def test_last_segment_of_one_atom():
    c = W.sc_cell(6, 6, 65, n_vac=143, jitter=0.05, seed=5)
    assert c.n == 9 * 1024 + 1
    _same(c, c, (1, 1, 1), noimage=True)


# cells with one, two and three shells of images along their shortest edge
@pytest.mark.parametrize("shape,vac,reps", [((4, 4, 4), 1, (1, 1, 1)), ((3, 4, 5), 2, (2, 1, 1)),
                                            ((2, 2, 2), 1, (2, 2, 2)), ((1, 3, 5), 1, (4, 2, 1))])
@pytest.mark.parametrize("wrapped", [True, False])
def test_image_lists(shape, vac, reps, wrapped):
    c = W.sc_cell(*shape, n_vac=vac, jitter=0.05, seed=7)
    big = _copies(c, reps)
    if not wrapped:  # images up to two cells away from an atom's own
        c.pos[:, ::3] += (np.asarray(c.lat).reshape(3, 3).diagonal() * [1, -2, 2])[:, None]
    _same(c, big, reps, noimage=True)


# k_relax_fire holds 1, 2 and 4 atoms a thread (1,008, 1,024 and 4,095 atoms,
# 4,096 the most); 4,097 atoms take the general state machine.  FP64 on both
# sides: the same number of steps and, over these few, the same positions to
# round-off (1e-9 A, as steps amplify the forces' 1e-10 eV/A by less than 10)
@pytest.mark.parametrize("shape,vac,final64", [
    ((4, 4, 4), 0, 0), ((6, 6, 7), 0, 0), ((8, 8, 4), 0, 0), ((8, 8, 16), 1, 0), ((8, 8, 16), 0, 0),
    ((5, 10, 21), 103, 0), ((6, 6, 7), 0, 1), ((5, 10, 21), 103, 1)])
def test_plain_fire_steps_match_oracle(oracle, shape, vac, final64):
    from akmc_amd import lib as L
    c = W.sc_cell(*shape, n_vac=vac, jitter=0.05, seed=9)
    steps = 12
    of = oracle.sc_field(["Cu"], ONE, 2 * CU["a"])
    cn = oracle.relax_defaults()
    cn.maxIter = steps
    o = oracle.fire_relax(oracle.FieldHandle(of, 0, c.types, c.lat), c.pos, cntrl=cn)
    f = L.Field(L.sc_potentials_text(ONE, 2 * CU["a"]))
    f.set_precision(64)
    b = L.Batch(f, [c])
    b.set_verify(16 if final64 else 0)
    b.start_relax(L.relax_defaults(maxIter=steps))
    b.run(4000, sync_every=5)
    st = b.status()[0]
    assert (st["status"], st["iterations"]) == (o["status"], o["iters"])
    dx = np.abs(W.min_image(b.positions()[0] - o["pos"], c.lat)).max()
    assert dx < 1e-9
    assert abs(st["energy"] - o["energy"]) < 1e-10 * abs(o["energy"])
