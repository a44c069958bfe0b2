"""PageRank over sizes where the propagation-blocked layout changes its widths
(rows per bin, columns per superblock)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the smallest width (256) and one past its range, whole and partial last
# bins, the edge of one round of superblocks (2^21) and of bins (2^22), where
# the narrow and wide scatter orders differ
SIZES = [1, 255, 257, 4096, 131072, 131073, 200003, (1 << 21) + 1, (1 << 22) + 1]


@pytest.mark.parametrize("n", SIZES)
def test_pb_layout_and_result_over_widths(tb, gpu, n):
    import torch
    c = 6 if n > 1 else 1
    m = tb.MatrixCSR().fill_cqmat_stochastic(n, n, c, 0.4, 11, device=True)
    from tbsla_amd._lib import check, lib
    check(lib.tbsla_hip_pb_layout_check(m._h))
    ref = torch.zeros(n, dtype=torch.float64, device="cuda")
    m.page_rank_device(ref, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="tiles")
    for precision in ("f64", "f32", "bf16", "pattern", "pattern_f32"):
        out = torch.zeros(n, dtype=torch.float64, device="cuda")
        m.page_rank_device(out, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="blocked",
                           precision=precision)
        # both are within 1e-10 (L1) of the fixed point
        assert float((out - ref).abs().sum()) <= 2e-10, precision
    out = torch.zeros(n, dtype=torch.float64, device="cuda")
    m.page_rank_device(out, epsilon=1e-8, max_iteration=500, gather="blocked")
    # the reference's rule stops at a step of 1e-8 of iterates of maximum 1 (so of sum >= 1): the rest of a
    # contraction by 0.85 is under 1e-8 * 0.85 / 0.15
    assert float((out - ref).abs().sum()) <= 1e-7
    assert np.isclose(float(out.sum()), 1.0, atol=1e-12)


@pytest.mark.parametrize("which", ["per_column", "first_differs", "last_differs", "last_bit_differs"])
def test_pb_column_values(tb, gpu, which):
    """Blocked products read no values where a column's entries agree; one entry that differs takes the stored
    values (a changed edge moves the vector far more than the bound)."""
    import torch
    n = 70001
    g = tb.MatrixCSR().fill_cqmat_stochastic(n, n, 6, 0.4, 5, device=True)
    a = g.arrays()
    ne = int(a["rowptr"][-1])
    col = a["colidx"][:ne]
    v = a["values"][:ne] * (0.5 + 0.5 * np.random.default_rng(3).random(n))[col]
    target = col[ne // 2]
    at = np.flatnonzero(col == target)
    assert at.size > 1
    if which == "first_differs":
        v[at[0]] *= 0.25
    elif which == "last_differs":
        v[at[-1]] *= 0.25
    elif which == "last_bit_differs":
        v[at[-1]] = np.nextafter(v[at[-1]], 1.0)
    m = tb.MatrixCSR(n, n, v, a["rowptr"], col)
    ref = torch.zeros(n, dtype=torch.float64, device="cuda")
    m.page_rank_device(ref, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="tiles")
    for precision in ("f64", "f32", "bf16"):
        out = torch.zeros(n, dtype=torch.float64, device="cuda")
        m.page_rank_device(out, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="blocked",
                           precision=precision)
        assert float((out - ref).abs().sum()) <= 2e-10, precision
    out = torch.zeros(n, dtype=torch.float64, device="cuda")
    m.page_rank_device(out, epsilon=1e-8, max_iteration=500, gather="blocked")
    assert float((out - ref).abs().sum()) <= 1e-7
