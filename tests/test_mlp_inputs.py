"""Shapes that MLP.train and MLP.predict take: rows of 48 inputs with 48
means and scales, what numpy broadcasts to that, and ValueError for anything
else before a pointer reaches the library."""
import numpy as np
import pytest

from akmc_amd import learn as LN
from akmc_amd import lib as L


@pytest.fixture
def net():
    LN._setup(L.load())
    m = LN.MLP.__new__(LN.MLP)  # no device: the library refuses the null handle
    m._h, m.max_rows = None, 256
    m.mean, m.scale = np.full(48, 0.5, np.float32), np.full(48, 2.0, np.float32)
    return m


@pytest.mark.parametrize("shape", [(5, 47), (5, 49), (5, 40), (48,), (0,), (2, 3, 48)])
def test_inputs_of_another_width_are_refused(net, shape):
    X = np.ones(shape, np.float32)
    with pytest.raises(ValueError):
        net.predict(X)
    with pytest.raises(ValueError):
        net.train(X, np.zeros((len(X), 3), np.float32), epochs=1)


@pytest.mark.parametrize("name", ["mean", "scale"])
@pytest.mark.parametrize("length", [1, 40, 47, 96])
def test_scaling_of_another_length(net, name, length):
    setattr(net, name, np.full(length, 0.25, np.float32))
    X = np.ones((5, 48), np.float32)
    if length == 1:  # broadcast
        Y, mean, scale = net._inputs(X)
        assert mean is None and scale is None and np.array_equal(Y, net.standardize(X))
    else:
        with pytest.raises(ValueError):
            net.predict(X)


def test_accepted_shapes_reach_the_library(net):
    X = np.ones((5, 48))
    Y, mean, scale = net._inputs(X)
    assert Y.dtype == np.float32 and mean is not None and scale is not None
    Y, mean, scale = net._inputs(np.ones((5, 1)))  # broadcast to 48 columns
    assert Y.shape == (5, 48) and mean is None and scale is None
    with pytest.raises(L.AkmcError):
        net.predict(X)
    with pytest.raises(ValueError):
        net.train(X, np.zeros((4, 3)), epochs=1)
