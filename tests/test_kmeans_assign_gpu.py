"""FP64 assignment on both sides of the line between one thread per row and the tile: 8,000 rows of
16 values meet at 13 centroids, 70,000 at 25 (24 of each 64 when there are more), 500,000 at 64."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,d,k", [(8_000, 15, 13), (8_000, 16, 14), (8_000, 40, 73), (70_000, 3, 25), (70_000, 17, 26),
                                   (70_000, 30, 72), (70_000, 33, 129), (70_000, 60, 24), (500_000, 9, 64),
                                   (500_000, 40, 64), (400_000, 40, 49)])
def test_labels(n, d, k, dtype):
    rng = np.random.default_rng(n + d + k)
    x = rng.normal(size=(n, d)).astype(dtype)
    c = x[rng.integers(0, n, k)].astype(np.float64)
    c[k // 2] = c[0]
    np.testing.assert_array_equal(S.kmeans_predict(x, c), O.kmeans_predict(x, c))
