"""Blocked PageRank where the gather reads the far products non-temporally: over
10 Mi of them in FP64 and 16 Mi in FP32, and up to 48 Mi."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,q", [(3000003, 8, 0.5), (5000011, 8, 0.5)])
def test_streamed_products(tb, gpu, n, c, q):
    """About 12 and 20 million far entries: FP64 alone streams, and both."""
    import torch
    m = tb.MatrixCSR().fill_cqmat_stochastic(n, n, c, q, 7, device=True)
    ref = torch.zeros(n, dtype=torch.float64, device="cuda")
    m.page_rank_device(ref, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="tiles")
    for precision in ("f64", "pattern", "f32", "bf16", "pattern_f32"):
        out = torch.zeros(n, dtype=torch.float64, device="cuda")
        m.page_rank_device(out, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="blocked",
                           precision=precision)
        # both are within 1e-10 (L1) of the fixed point
        assert float((out - ref).abs().sum()) <= 2e-10, precision
    m.page_rank_device(out, epsilon=1e-8, max_iteration=500, gather="blocked")
    # a step of 1e-8 of iterates of sum >= 1 leaves under 1e-8 * 0.85 / 0.15
    assert float((out - ref).abs().sum()) <= 1e-7


def test_streamed_stored_values(tb, gpu):
    import numpy as np
    import torch
    n = 5000011
    a = tb.MatrixCSR().fill_cqmat_stochastic(n, n, 8, 0.5, 7, device=True).arrays()
    v = a["values"] * (0.5 + 0.5 * np.random.default_rng(1).random(a["values"].size))
    m = tb.MatrixCSR(n, n, v, a["rowptr"], a["colidx"])
    ref, out = (torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(2))
    m.page_rank_device(ref, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="tiles")
    for precision in ("f64", "f32", "bf16"):
        m.page_rank_device(out, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="blocked",
                           precision=precision)
        assert float((out - ref).abs().sum()) <= 2e-10, precision
