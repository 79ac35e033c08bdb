"""The network's outputs for host rows around the sizes where they leave by
another way: the output layer's own stores into pinned memory up to 1024 rows,
a copy above.  A row's outputs do not depend on the others."""
import numpy as np
import pytest

import brownian_amd as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 33, 1023, 1024, 1025, 2000])
def test_rows_do_not_depend_on_the_batch(n):
    rng = np.random.default_rng(7)
    net = B.MLP(seed=2)
    x = rng.normal(size=(2000, 144)).astype(np.float32)
    whole = net.forward(x)
    y = net.forward(x[:n])
    assert y.shape == (n, 12) and np.isfinite(y).all() and np.abs(y).max() > 0
    np.testing.assert_array_equal(y, whole[:n])
