"""PageRank on small graphs with long rows, around the length from which they are
not one workgroup's, against the oracle: 64 loads of eight entries in one
wavefront (a row of 512, or rows of 256 and less in several rounds of 1024)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows", [(700, {5: 512}), (700, {5: 513}), (700, {0: 512, 64: 512, 699: 505}),
                                    (2100, {3: 256, 1027: 248, 2051: 8}), (2100, {3: 256, 1027: 256, 2051: 8}),
                                    (5632, {5631: 400}), (5632, {5631: 900})])
@pytest.mark.parametrize("per_column", [True, False])
def test_long_rows(tb, oracle, gpu, n, rows, per_column):
    rng = np.random.default_rng(n)
    lens = rng.integers(0, 4, n)
    for r, k in rows.items():
        lens[r] = k
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = rng.integers(0, n, ptr[-1]).astype(np.int32)
    val = (1.0 / np.maximum(np.bincount(col, minlength=n), 1))[col]
    if not per_column:
        val = val * (0.5 + 0.5 * rng.random(val.size))
    m = tb.MatrixCSR(n, n, val, ptr, col)
    o = oracle.from_arrays("CSR", n, n, val, ptr, col)
    got, it = m.page_rank(1e-9, 0.85, 200)
    want, jt = o.page_rank(1e-9, 0.85, 200)
    # the same left-to-right row sums; only the order of the residual's and the sum's additions differs
    assert abs(it - jt) <= 1 and np.abs(got - want).sum() <= 1e-12
