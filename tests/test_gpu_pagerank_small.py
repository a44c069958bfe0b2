"""PageRank on graphs that one workgroup runs in one launch, against the
oracle: sizes around the row count of a round of threads and the largest
that fits, entries read with and without values, rows longer than a chunk,
the longest row it takes and one more, and runs of several launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def close(got, it, want, jt):
    # the same left-to-right row sums; only the order of the residual's and the sum's additions differs
    assert abs(it - jt) <= 1 and np.abs(got - want).sum() <= 1e-12, (it, jt, np.abs(got - want).sum())


@pytest.mark.parametrize("n", [1, 2, 63, 1023, 1024, 1025, 2049, 5631, 5632, 5633])
@pytest.mark.parametrize("c", [3, 11])
def test_sizes(tb, oracle, gpu, n, c):
    c = min(c, n)
    m = tb.MatrixCSR().fill_cqmat_stochastic(n, n, c, 0.4, 7)
    o = oracle.new("CSR").fill_cqmat_stochastic(n, n, c, 0.4, 7)
    close(*m.page_rank(1e-9, 0.85, 200), *o.page_rank(1e-9, 0.85, 200))
    nodes = np.unique(np.array([0, n // 2, n - 1], dtype=np.int32))
    close(*m.personalized_page_rank(1e-9, 0.85, 200, nodes), *o.personalized_page_rank(1e-9, 0.85, 200, nodes))


@pytest.mark.parametrize("longest", [9, 17, 1536, 1537])
@pytest.mark.parametrize("per_column", [True, False])
def test_row_lengths_and_values(tb, oracle, gpu, longest, per_column):
    n = 2000
    rng = np.random.default_rng(longest)
    lens = rng.integers(0, 9, n)
    lens[[0, 700, n - 1]] = longest
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = rng.integers(0, n, ptr[-1]).astype(np.int32)
    cnt = np.bincount(col, minlength=n)
    val = (1.0 / np.maximum(cnt, 1))[col]
    if not per_column:
        val = val * (0.5 + 0.5 * rng.random(val.size))
    m = tb.MatrixCSR(n, n, val, ptr, col)
    o = oracle.from_arrays("CSR", n, n, val, ptr, col)
    close(*m.page_rank(1e-9, 0.85, 200), *o.page_rank(1e-9, 0.85, 200))


def test_several_launches(tb, gpu):
    import torch
    n = 1500
    m = tb.MatrixCSR().fill_cqmat_stochastic(n, n, 6, 0.4, 7)
    a, b = (torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(2))
    for most in (255, 256, 257, 600):
        r = m.page_rank_device(a, epsilon=0.0, max_iteration=most, gather="tiles")
        assert r["iterations"] == most
    r = m.page_rank_device(b, epsilon=0.0, max_iteration=256, gather="tiles", teleport=torch.full_like(b, 1.0 / n))
    assert r["iterations"] == 256 and float((a - b).abs().sum()) <= 1e-12
