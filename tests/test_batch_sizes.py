"""Batched PageRank over the sizes where its passes have edges: groups of 2,
63, 64 and 65 sets on graphs of less than, equal to and just over 64 rows and
1024 rows, stopped after even and odd iteration counts, against the same sets
one at a time (which run as single-set graphs)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1025, 2048, 2049])
@pytest.mark.parametrize("k", [2, 63, 64, 65])
def test_group_equals_single_sets(tb, gpu, n, k):
    m = tb.MatrixCSR().fill_cqmat_stochastic(n, n, min(n, 5), 0.4, 3)
    sets = [[(17 * r) % n] for r in range(k)]
    for precision, tol in (("f64", 1e-13), ("f32", 1e-5)):
        for most in (0, 1, 2, 7):
            g = tb.PageRankBatch(precision).add_graph(m, sets)
            s = tb.PageRankBatch(precision)
            for nodes in sets:
                s.add_graph(m, [nodes])
            a, _, ia = g.run(epsilon=1e-30, max_iteration=most, rule="sumnorm")
            b, _, ib = s.run(epsilon=1e-30, max_iteration=most, rule="sumnorm")
            assert np.array_equal(ia, ib)
            d = (a - b).abs().reshape(k, n).sum(1)
            assert float(d.max()) <= tol, (precision, most, float(d.max()))
