"""The candidate store of a search that runs in batches of queries has to hold every batch: a short
last batch spreads over more pieces and may need more entries than the full ones."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# Every batch's entries and lists against the store, over a range of searches; prints the number of
# searches whose last batch is the largest.
CHECK = r"""
#include "knn_lists.hpp"
#include <cstdio>
using namespace sc;
int main() {
  int larger = 0;
  for (int tile : {128, 32})
    for (int k : {1, 10, 64})
      for (int64_t n : {1500, 20000, 300000, 4000000})
        for (int64_t q = 1; q < 200000; q = q * 5 / 4 + 37) {
          const std::vector<int64_t> edge = level_edges(n, std::min<int64_t>(kDenseRows, (n + 127) / 128 * 128));
          auto plan = [&](int64_t qn, Level (&lv)[kMaxLevels], ScanOut<double>& o) {
            plan_levels(edge, qn, qn <= 32 ? tile : 128, 512, k, lv, o);
          };
          Level lv[kMaxLevels];
          ScanOut<double> o{};
          const auto b = plan_batches(q, plan, [&](const ScanOut<double>& p) { return 12.0 * p.entries + 4.0 * p.lists; }, lv, o);
          if (o.entries * b.queries > b.entries || o.lists * b.queries > b.lists) return 1;
          const int64_t first = o.entries * b.queries;
          for (int64_t b0 = 0; b0 < q; b0 += b.queries) {
            const int64_t qn = std::min(b.queries, q - b0);
            plan(qn, lv, o);
            if (o.entries * qn > b.entries || o.lists * qn > b.lists) return 2;
            larger += o.entries * qn > first;
          }
        }
  std::printf("%d\n", larger);
}
"""


def test_store_holds_every_batch(tmp_path):
    src, exe = tmp_path / "check.hip", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-host-only", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "smartcore_amd", "csrc"), str(src), "-o", str(exe)], check=True,
                   capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0
    assert int(r.stdout) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("metric,n,q,k", [("euclidian", 300_000, 132_178, 10), ("manhattan", 20_000, 55_846, 20)])
def test_batches_equal_single_searches(metric, n, q, k):
    """Searches of several batches with the largest one last, against searches of one batch each and
    the oracle."""
    import oracle as O
    from smartcore_amd import _capi as S

    rng = np.random.default_rng(n + q)
    x, y = rng.normal(size=(n, 2)).astype(np.float32), rng.normal(size=(q, 2)).astype(np.float32)
    m, mode, om = ((S.SC_EUCLIDIAN, S.SC_PLAIN_FP64, O.EUCLIDIAN) if metric == "euclidian" else
                   (S.SC_MANHATTAN, S.SC_MIXED, O.MANHATTAN))
    ix = S.Index(x)
    gi, gd, gc = ix.knn(y, k, m, 2, mode)
    assert (gc == k).all()
    for a in range(0, q, 5_000):
        pi, pd, _ = ix.knn(y[a:a + 5_000], k, m, 2, mode)
        np.testing.assert_array_equal(gi[a:a + 5_000], pi)
        np.testing.assert_array_equal(gd[a:a + 5_000].view(np.uint64), pd.view(np.uint64))
    for r in (0, q // 2, q - 1):
        oi, od = O.linear_find(x, y[r], k, om)
        np.testing.assert_array_equal(gi[r], oi)
        np.testing.assert_array_equal(gd[r].view(np.uint64), np.asarray(od).view(np.uint64))
