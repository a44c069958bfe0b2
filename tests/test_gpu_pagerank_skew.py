"""Blocked PageRank where the two scatter orders differ (over 2^21 nodes) and the
columns are even, or crowd into the first superblocks: value-free products then
take the wide order, or the narrow one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("power", [1.0, 2.0])
@pytest.mark.parametrize("per_column", [True, False])
def test_crowded_columns(tb, gpu, power, per_column):
    import torch
    from tbsla_amd._lib import check, lib
    n, c = (1 << 21) + 4097, 4
    rng = np.random.default_rng(4)
    col = np.minimum((n * rng.random(n * c) ** power).astype(np.int64), n - 1).astype(np.int32)
    v = (1.0 / np.maximum(np.bincount(col, minlength=n), 1))[col]
    if not per_column:
        v = v * (0.5 + 0.5 * rng.random(v.size))
    m = tb.MatrixCSR(n, n, v, (np.arange(n + 1) * c).astype(np.int32), col)
    check(lib.tbsla_hip_pb_layout_check(m._h))
    ref, out = (torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(2))
    m.page_rank_device(ref, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="tiles")
    for precision in ("f64", "f32", "bf16"):
        m.page_rank_device(out, epsilon=1e-10, max_iteration=500, rule="sumnorm", gather="blocked",
                           precision=precision)
        # both are within 1e-10 (L1) of the fixed point
        assert float((out - ref).abs().sum()) <= 2e-10, precision
    m.page_rank_device(out, epsilon=1e-8, max_iteration=500, gather="blocked")
    # a step of 1e-8 of iterates of sum >= 1 leaves under 1e-8 * 0.85 / 0.15
    assert float((out - ref).abs().sum()) <= 1e-7
