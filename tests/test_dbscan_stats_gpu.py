"""The row pairs that a DBSCAN fit computes: all tile pairs of a small set, those of the near tiles
only of a large one."""
import numpy as np
import pytest

from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def test_pairs_computed():
    rng = np.random.default_rng(3)
    S.Index(rng.normal(size=(300, 3))).dbscan_fit(0.5, 5)  # three tiles: six pairs of tiles
    assert S.last_stats()["queries"] == 300 and S.last_stats()["candidates"] == 6 * 128 * 128
    far = rng.normal(size=(40_000, 3)) + 1e4 * rng.integers(0, 40, size=(40_000, 1))
    S.Index(far).dbscan_fit(0.5, 5)
    assert 40_000 <= S.last_stats()["candidates"] < 40_000 ** 2 // 4
