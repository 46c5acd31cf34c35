"""Distances of one query to listed rows on the host, at the row lengths where
more or fewer rows are taken together and for every number left over: bit for
bit the oracle's."""
import numpy as np
import pytest

import oracle
from pilotann_amd import _lib


@pytest.mark.parametrize('d', [8, 184, 192, 200])
def test_rows_taken_together(d):
    rng = np.random.default_rng(d)
    storage = rng.standard_normal((300, d), dtype=np.float32)
    query = rng.standard_normal(d, dtype=np.float32)
    for n in [*range(1, 18), 63, 64, 65, 130]:
        nodes = rng.integers(0, 300, n)
        out = np.full(n + 1, 7.0, np.float32)
        _lib.check(_lib.lib().pa_square_dist(
            out.ctypes.data, query.ctypes.data, storage.ctypes.data, nodes.ctypes.data, n, 300,
            d), 'pa_square_dist')
        assert np.array_equal(out[:n], oracle.square_dist(query, storage, nodes))
        assert out[n] == 7.0
