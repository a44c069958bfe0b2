"""Mixed-precision PageRank on the entry tiles over the sizes where the sum of its
result is split differently: less than a block of 1024 nodes, one and a few,
more than 512, and more than one step of eight nodes a thread."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1000, 1025, 600001, (1 << 22) + 5])
def test_sum_of_mixed_tile_results(tb, gpu, n):
    import torch
    m = tb.MatrixCSR().fill_cqmat_stochastic(n, n, min(n, 6), 0.4, 11, device=True)
    ref = torch.zeros(n, dtype=torch.float64, device="cuda")
    m.page_rank_device(ref, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="tiles")
    for precision in ("f32", "bf16", "pattern_f32"):
        out = torch.zeros(n, dtype=torch.float64, device="cuda")
        m.page_rank_device(out, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="tiles", precision=precision)
        # both are within 1e-10 (L1) of the fixed point, of sum 1 up to the roundings of n quotients
        assert float((out - ref).abs().sum()) <= 2e-10, precision
        assert abs(float(out.sum()) - 1.0) <= 1e-12, precision
