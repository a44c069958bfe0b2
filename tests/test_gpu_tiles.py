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


@pytest.mark.parametrize("fmt", ["CSR", "COO"])
@pytest.mark.parametrize("shortest,longest,rows", [(0, 40, 9000), (100, 256, 1500), (256, 257, 900), (200, 600, 400),
                                                   (1100, 1536, 130), (1500, 1540, 40)])
def test_rows_past_their_tile_exact(tb, oracle, gpu, fmt, shortest, longest, rows):
    """Rows of every offset from their tile's end: what is staged of them beside
    the tile, and what the block stages after it.  Rows over 1536 entries are
    tree sums, within 1e-13 of sum |a||x| (fewer than 30 roundings a product)."""
    rng = np.random.default_rng(longest)
    lens = rng.integers(shortest, longest + 1, rows)
    n = max(rows, 1600)
    row = np.repeat(np.arange(rows, dtype=np.int32), lens)
    col = rng.integers(0, n, row.size).astype(np.int32)
    val, x = rng.random(row.size) - 0.5, rng.random(n) - 0.5
    # (both hold the entries in this order; a conversion would sort the columns)
    ptr = np.concatenate([[0], np.cumsum(lens), np.full(n - rows, row.size)]).astype(np.int32)
    m = tb.MatrixCOO(n, n, val, row, col) if fmt == "COO" else tb.MatrixCSR(n, n, val, ptr, col)
    o = oracle.from_arrays("COO", n, n, val, row, col)
    y, yo = m.spmv(x), o.spmv(x)
    exact = np.concatenate([lens <= 1536, np.ones(n - rows, bool)])
    assert np.array_equal(y[exact], yo[exact])
    absy = oracle.from_arrays("COO", n, n, np.abs(val), row, col).spmv(np.abs(x))
    assert np.all(np.abs(y - yo) <= 1e-13 * absy)
