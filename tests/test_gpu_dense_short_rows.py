"""Dense products over the row lengths where the lanes' share of a row changes:
one column a lane up to 192 columns, two from there on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 5, 7171])
@pytest.mark.parametrize("cols", [2, 63, 64, 65, 128, 191, 192, 193, 194])
def test_dense_short_rows(tb, gpu, rows, cols):
    """Each row within 1e-14 of sum |a||x|: a product passes at most 4 sums in its lane and 6 in the butterfly, 11
    roundings or 1.3e-15; numpy's product stays under 194 * 2^-53 = 2.2e-14 / 8 lanes."""
    rng = np.random.default_rng(rows + cols)
    a = rng.random((rows, cols)) - 0.5
    r, c = np.indices((rows, cols), dtype=np.int32)
    m = tb.MatrixDENSE(tb.MatrixCOO(rows, cols, a.ravel(), r.ravel(), c.ravel()))
    x = rng.random(cols) - 0.5
    assert np.all(np.abs(m.spmv(x) - a @ x) <= 1e-14 * (np.abs(a) @ np.abs(x)))
