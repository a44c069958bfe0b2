"""Blocked PageRank on graphs whose edges stay near their row, over the shares of
local entries (column in the row's bin) where the gather changes how it reads
them: columns beside each other and apart, most, some and few of them local,
bins whole and partial."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def window_graph(tb, n, c, w, per_column=True):
    """c columns a row, within w of it (w = 0: the c columns from it on)."""
    rng = np.random.default_rng(w + c)
    base = np.repeat(np.arange(n, dtype=np.int64), c)
    off = np.tile(np.arange(c), n) if w == 0 else rng.integers(-w, w + 1, base.size)
    col = np.sort(((base + off) % n).reshape(n, c), axis=1).ravel().astype(np.int32)
    v = (1.0 / np.maximum(np.bincount(col, minlength=n), 1))[col]
    if not per_column:
        v = v * (0.5 + 0.5 * rng.random(v.size))
    return tb.MatrixCSR(n, n, v, (np.arange(n + 1) * c).astype(np.int32), col)


@pytest.mark.parametrize("n", [300, 66000, 70001])
@pytest.mark.parametrize("c,w", [(5, 0), (8, 60), (8, 150), (8, 400), (8, 900), (8, 30000)])
def test_local_entries(tb, gpu, n, c, w):
    import torch
    from tbsla_amd._lib import check, lib
    m = window_graph(tb, n, c, w)
    check(lib.tbsla_hip_pb_layout_check(m._h))
    nodes = [0, n // 2, n - 1]
    for kw in ({}, {"nodes": nodes}, {"teleport": torch.linspace(0.5, 1.5, n, dtype=torch.float64, device="cuda") / n}):
        ref, out = (torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(2))
        m.page_rank_device(ref, epsilon=1e-11, max_iteration=900, rule="sumnorm", gather="tiles", **kw)
        m.page_rank_device(out, epsilon=1e-11, max_iteration=900, rule="sumnorm", gather="blocked", **kw)
        # both are within 1e-11 (L1) of the fixed point
        assert float((out - ref).abs().sum()) <= 2e-11, kw
        m.page_rank_device(out, epsilon=1e-8, max_iteration=900, gather="blocked", **kw)
        # a step of 1e-8 of iterates of sum >= 1 leaves under 1e-8 * 0.85 / 0.15
        assert float((out - ref).abs().sum()) <= 1e-7, kw
