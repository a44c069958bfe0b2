"""Products over both column widths of the device mirrors (three bytes up to
2^24 columns, else four) with every remainder of a group of four: rows are the
left-to-right sums of the stored entries, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def row_sums(n, row, col, val, x):
    y = np.zeros(n)
    for r, c, v in zip(row, col, val):
        y[r] += float(v) * float(x[c])
    return y


@pytest.mark.parametrize("fmt", ["CSR", "SCOO", "COO", "ELL"])
@pytest.mark.parametrize("last", [(1 << 24) - 1, 1 << 24])
def test_columns_at_the_packed_limit(tb, gpu, fmt, last):
    n, n_col, k = 37, (1 << 24) + 9, 7
    rng = np.random.default_rng(last)
    col = np.sort(rng.choice(last, (n, k), replace=False), axis=1).astype(np.int32)
    col[5, k - 1] = last
    row = np.repeat(np.arange(n, dtype=np.int32), k)
    val = rng.random(n * k)
    x = rng.random(n_col)
    coo = tb.MatrixCOO(n, n_col, val, row, col.ravel())
    m = coo if fmt == "COO" else tb.FORMATS[fmt](coo)
    assert np.array_equal(m.spmv(x), row_sums(n, row, col.ravel(), val, x))


@pytest.mark.parametrize("fmt", ["CSR", "SCOO"])
@pytest.mark.parametrize("rows", [146, 147, 1000])
@pytest.mark.parametrize("n_col", [450_000, 600_001, (1 << 24) + 9])
def test_whole_tiles_against_a_large_x(tb, gpu, fmt, rows, n_col):
    """1022, 1029 and 7000 entries: no, one and several whole tiles, with an x
    that stays in an L2 and with ones that do not."""
    k = 7
    rng = np.random.default_rng(rows)
    col = np.sort(rng.integers(0, n_col, (rows, k)), axis=1).astype(np.int32)
    col[rows // 2, k - 1] = n_col - 1
    row = np.repeat(np.arange(rows, dtype=np.int32), k)
    val = rng.random(rows * k)
    x = rng.random(n_col)
    m = tb.FORMATS[fmt](tb.MatrixCOO(rows, n_col, val, row, col.ravel()))
    assert np.array_equal(m.spmv(x), row_sums(rows, row, col.ravel(), val, x))


@pytest.mark.parametrize("fmt", ["CSR", "SCOO", "ELL"])
@pytest.mark.parametrize("k", list(range(1, 10)) + [16, 19])
@pytest.mark.parametrize("n", [19, 64, 255, 257, 1000])
def test_column_groups_exact(tb, oracle, gpu, fmt, k, n):
    m = tb.FORMATS[fmt]().fill_cqmat(n, n, k, 0.3, 5, value_seed=5)
    x = oracle.uniform_vector(1, n)
    o = oracle.new(fmt).fill_cqmat(n, n, k, 0.3, 5, value_seed=5)
    assert np.array_equal(m.spmv(x), o.spmv(x))
