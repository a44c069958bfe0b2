"""Dense products over rows of odd and even length, below and from the row count
where wavefronts take four rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 2), (5, 127), (9, 128), (6, 129), (7, 255), (33, 256), (10, 257),
                                       (257, 513), (7167, 130), (7168, 131), (7171, 383)])
def test_dense_row_lengths(tb, gpu, rows, cols):
    """Each row within 1e-14 of sum |a||x|: a product passes at most 2 * 3 sums
    in its lane (513 columns) and 6 in the butterfly, 13 roundings or 1.5e-15;
    numpy's product stays under 513 * 2^-53 / 8 = 7e-15."""
    rng = np.random.default_rng(rows + cols)
    a = rng.random((rows, cols)) - 0.5
    r, c = np.indices((rows, cols), dtype=np.int32)
    m = tb.MatrixDENSE(tb.MatrixCOO(rows, cols, a.ravel(), r.ravel(), c.ravel()))
    x = rng.random(cols) - 0.5
    assert np.all(np.abs(m.spmv(x) - a @ x) <= 1e-14 * (np.abs(a) @ np.abs(x)))
