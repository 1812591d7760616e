"""Ward's rounds against the same rounds over all pairs.

The GPU's clusters keep lists of their nearest and search again only when merged
or out of entries; every nearest, ties included, is to be the one that a pass
over all pairs finds. The reference runs those passes on the host (compiled with
g++; skipped when it is absent): FP32 Ward weights of FP32-rounded centroids, the
lowest (weight, slot), merges of reciprocal pairs in FP64. Every operation is
correctly rounded on both sides, so the trees are equal bit for bit.
"""

import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

import cuhc_amd as cuhc
from _helpers import assert_same_dendrogram
from cuhc_amd import _lib
from cuhc_amd._linkage import _ward_rnn_with_options

pytestmark = pytest.mark.gpu
CSRC = Path(__file__).resolve().parent.parent / "cuhc_amd" / "csrc"

DRIVER = r"""
#include "host_tree.hpp"
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
using cuhc::Edge;
// argv: points file (float32), n, d, tree file (float64).
int main(int, char **argv) {
  const int n = std::atoi(argv[2]), d = std::atoi(argv[3]);
  std::vector<float> x((size_t)n * d);
  FILE *f = std::fopen(argv[1], "rb");
  if (!f || std::fread(x.data(), sizeof(float), x.size(), f) != x.size())
    return 1;
  std::fclose(f);
  std::vector<double> c(x.begin(), x.end());
  std::vector<int> size(n, 1), rep(n), nearest(n);
  for (int i = 0; i < n; ++i)
    rep[i] = i;
  std::vector<Edge> all;
  for (int m = n; m > 1;) {
    for (int i = 0; i < m; ++i) {
      float best = INFINITY;
      nearest[i] = -1;
      for (int j = 0; j < m; ++j) {
        if (j == i)
          continue;
        float sq = 0.0f;
        for (int k = 0; k < d; ++k) {
          const float diff = x[(size_t)i * d + k] - x[(size_t)j * d + k];
          sq = std::fma(diff, diff, sq);
        }
        const float si = (float)size[i], sj = (float)size[j];
        const float w = (2.0f * (si * sj)) / (si + sj) * sq;
        if (w < best) { // the lowest slot of equal weights
          best = w;
          nearest[i] = j;
        }
      }
    }
    const size_t first = all.size();
    int at = 0;
    for (int i = 0; i < m; ++i) {
      const int j = nearest[i];
      const bool pair = j >= 0 && nearest[j] == i;
      if (pair && j < i)
        continue;
      int newSize = size[i];
      if (pair) {
        const double si = size[i], sj = size[j];
        double sq = 0.0;
        for (int k = 0; k < d; ++k) {
          const double ci = c[(size_t)i * d + k], cj = c[(size_t)j * d + k];
          sq = std::fma(ci - cj, ci - cj, sq);
        }
        all.push_back(Edge{std::min(rep[i], rep[j]), std::max(rep[i], rep[j]),
                           std::sqrt(2.0 * (si * sj) / (si + sj) * sq)});
        for (int k = 0; k < d; ++k) {
          const double ci = c[(size_t)i * d + k];
          c[(size_t)i * d + k] = std::fma(c[(size_t)j * d + k] - ci, sj / (si + sj), ci);
        }
        newSize += size[j];
      }
      for (int k = 0; k < d; ++k) {
        c[(size_t)at * d + k] = c[(size_t)i * d + k];
        x[(size_t)at * d + k] = (float)c[(size_t)at * d + k];
      }
      rep[at] = rep[i];
      size[at] = newSize;
      ++at;
    }
    if (at == m)
      return 2;
    m = at;
    std::sort(all.begin() + first, all.end(), cuhc::edgeLess);
  }
  std::vector<double> tree((size_t)(n - 1) * 4);
  if (!cuhc::mergesToTreeOrder(all, n))
    return 3;
  cuhc::treeFromOrderedMerges(all, n, tree.data());
  f = std::fopen(argv[4], "wb");
  return f && std::fwrite(tree.data(), sizeof(double), tree.size(), f) == tree.size() &&
                 std::fclose(f) == 0 ? 0 : 4;
}
"""


@pytest.fixture(scope="module")
def reference(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    folder = tmp_path_factory.mktemp("ward_rounds")
    (folder / "driver.cpp").write_text(DRIVER)
    subprocess.run([gxx, "-O3", "-std=c++17", "-mfma", "-ffp-contract=off", "-I", str(CSRC),
                    str(folder / "driver.cpp"), str(CSRC / "host_tree.cpp"),
                    str(CSRC / "extract.cpp"), "-o", str(folder / "driver")],
                   check=True, capture_output=True, text=True)

    def tree(X):
        X.astype(np.float32).tofile(folder / "points")
        subprocess.run([str(folder / "driver"), str(folder / "points"), *map(str, X.shape),
                        str(folder / "tree")], check=True)
        return np.fromfile(folder / "tree").reshape(-1, 4)

    return tree


@pytest.mark.parametrize("n, d, values", [(65, 2, 6), (700, 2, 6), (2100, 2, 40), (900, 17, 3),
                                          (1300, 33, 2), (1500, 7, None), (8200, 3, 25),
                                          (16_500, 3, 60)])
def test_lists_find_what_a_pass_over_all_pairs_finds(reference, n, d, values):
    # Integer lattices (values per feature): most weights tie, lists end in
    # equal keys, offers tie with bounds and lists run out. 17 and 33 features:
    # first lists from the mixed pass; above 8,192 clusters the rounds are
    # numbered by a scan, above 16,384 searches take tiles of 128.
    rng = np.random.default_rng(n + d)
    X = rng.integers(0, values, (n, d)) if values else rng.normal(size=(n, d))
    X = X.astype(np.float32)
    Z = _ward_rnn_with_options(X, min_progress=0.0, allow_dense=False)
    np.testing.assert_array_equal(Z, reference(X))


@pytest.mark.parametrize("d, pruning", [(5, "never"), (33, "never"), (70, "never"),
                                        (20, "always")])
def test_wide_search_tiles_against_the_chain(d, pruning):
    # Searches of tiles of 128 over one fill of 8 features and over one, two and
    # three fills of 32, the first of them of all rows; and lists of one key from
    # a pruned pass that gives up above that size.
    X = np.random.default_rng(d).normal(size=(16_700, d)).astype(np.float32)
    _lib.set_precision("fp32")
    _lib.set_pruning(pruning)
    try:
        rnn = cuhc.linkage(X, method="ward", algorithm="rnn")
    finally:
        _lib.set_precision("auto")
        _lib.set_pruning("auto")
    chain = cuhc.linkage(X, method="ward", algorithm="nn_chain")
    assert_same_dendrogram(rnn, chain, rtol=1e-5, atol=1e-6)
