"""PageRank on the entry tiles of graphs with long rows: staged past their tile (up
to 1536 entries), summed by a workgroup of their own (more), and both, with the
step decision merged into the update (up to 2^20 entries) and apart, against the
oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,base", [(6000, 4), (60000, 8), (60000, 20)])
@pytest.mark.parametrize("hubs", [[257], [1536, 1024], [1537], [5000, 600, 1300]])
def test_hub_rows(tb, oracle, gpu, n, base, hubs):
    rng = np.random.default_rng(n + len(hubs))
    lens = rng.integers(0, base, n)
    lens[rng.choice(n, len(hubs), replace=False)] = hubs
    lens[n - 1] = hubs[0]
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = rng.integers(0, n, ptr[-1]).astype(np.int32)
    val = (1.0 / np.maximum(np.bincount(col, minlength=n), 1))[col] * (0.5 + 0.5 * rng.random(col.size))
    m = tb.MatrixCSR(n, n, val, ptr, col)
    o = oracle.from_arrays("CSR", n, n, val, ptr, col)
    # the same row sums but for rows over 1536 entries (a tree); else only the order of the residual's and the sum's
    # additions differs
    got, it = m.page_rank(1e-9, 0.85, 200)
    want, jt = o.page_rank(1e-9, 0.85, 200)
    assert abs(it - jt) <= 1 and np.abs(got - want).sum() <= 1e-12
    nodes = np.array([0, n // 2, n - 1], dtype=np.int32)
    got, it = m.personalized_page_rank(1e-9, 0.85, 200, nodes)
    want, jt = o.personalized_page_rank(1e-9, 0.85, 200, nodes)
    assert abs(it - jt) <= 1 and np.abs(got - want).sum() <= 1e-12
