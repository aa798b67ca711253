"""An index whose preparation has 2^32 threads and more when each row takes several: past what one
launch holds.  Every search that prepares rows must answer as the oracle does."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def test_searches_over_half_a_billion_rows():
    n = (1 << 29) + 1_000  # eight lanes a row: 2^32 threads (sixteen: from 2^28 rows on)
    host = np.random.default_rng(5).random((n, 1), dtype=np.float32)
    host += 50.0
    near = [0, 7, 300, 900, n // 2, n - 900, n - 2, n - 1]  # every other row is at least 48 away
    host[near, 0] = [1.9, 1.1, 1.7, 0.9, 1.3, 0.2, 1.5, 0.6]
    ix = S.Index(host)
    qs = np.array([[0.0], [1.45]], np.float32)
    for metric, mode, om in ((S.SC_EUCLIDIAN, S.SC_PLAIN_FP64, O.EUCLIDIAN), (S.SC_EUCLIDIAN, S.SC_MIXED, O.EUCLIDIAN),
                             (S.SC_MANHATTAN, S.SC_MIXED, O.MANHATTAN)):
        gi, gd, gc = ix.knn(qs, 4, metric, 2, mode)
        for r, y in enumerate(qs):
            oi, od = O.linear_find(host, y, 4, om)
            assert gc[r] == 4
            np.testing.assert_array_equal(gi[r], oi)
            np.testing.assert_array_equal(gd[r].view(np.uint64), np.asarray(od).view(np.uint64))
    for r, (rows, dist) in enumerate(ix.radius(qs, 1.0)):
        oi, od = O.linear_find_radius(host, qs[r], 1.0, O.EUCLIDIAN)
        np.testing.assert_array_equal(rows, oi)
        np.testing.assert_array_equal(dist.view(np.uint64), od.view(np.uint64))
