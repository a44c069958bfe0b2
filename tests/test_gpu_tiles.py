"""Products over the sizes where the entry tiles change: whole and partial
tiles of 1024 entries, the step to 2048 entries past 2^20, and rows of 256
entries (the longest with small tiles) and 257.  Every row is the reference's
left-to-right sum, so the results are equal bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["CSR", "SCOO", "COO"])
@pytest.mark.parametrize("n,c", [(1, 1), (128, 8), (129, 8), (1024, 3), (65536, 16), (65600, 16), (66000, 16)])
def test_tile_sizes_exact(tb, oracle, gpu, fmt, n, c):
    m = tb.FORMATS[fmt]().fill_cqmat(n, n, c, 0.25, 9, value_seed=9)
    x = oracle.uniform_vector(1, n)
    o = oracle.new("CSR").fill_cqmat(n, n, c, 0.25, 9, value_seed=9)
    assert np.array_equal(m.spmv(x), o.spmv(x))


@pytest.mark.parametrize("longest", [256, 257])
def test_rows_over_small_tiles_exact(tb, gpu, longest):
    rng = np.random.default_rng(longest)
    lens = np.full(3000, 3)
    lens[[0, 7, 500, 2999]] = longest
    lens[[3, 4]] = 0
    ptr = np.concatenate([[0], np.cumsum(lens)])
    col = rng.integers(0, 3000, ptr[-1])
    val, x = rng.random(ptr[-1]), rng.random(3000)
    y = tb.MatrixCSR(3000, 3000, val, ptr, col).spmv(x)
    for r in (0, 1, 3, 6, 7, 8, 500, 501, 1700, 2998, 2999):
        s = 0.0
        for k in range(ptr[r], ptr[r + 1]):
            s += float(val[k]) * float(x[col[k]])
        assert y[r] == s, r
