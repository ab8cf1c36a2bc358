"""predict on both sides of the row count up to which inputs are standardised
on the host: the bits of forward on rows standardised by numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 47, 1024, 1025, 4097])
def test_predict_equals_forward_of_standardised_rows(rows):
    from akmc_amd import learn as LN
    rng = np.random.default_rng(rows)
    X = (3 * rng.standard_normal((rows, 48)) + 1).astype(np.float32)
    m = LN.MLP(max_rows=2048, seed=1)
    m.mean = rng.standard_normal(48).astype(np.float32)
    m.scale = rng.uniform(0.1, 3, 48).astype(np.float32)
    assert np.array_equal(m.predict(X), m.forward(m.standardize(X)))
