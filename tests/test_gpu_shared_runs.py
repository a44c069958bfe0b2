"""PageRank runs with blocked products in flight together on one matrix, from
several threads and streams: the layout is shared, the products are not."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BLOCKED = [{"rule": "sumnorm", "precision": "f64"}, {"rule": "sumnorm", "precision": "f32"},
           {"rule": "sumnorm", "precision": "bf16"}, {"rule": "reference", "precision": "f64"},
           {"rule": "sumnorm", "precision": "f64", "nodes": [3, 99]}]


@pytest.mark.parametrize("per_column", [True, False])
def test_threads_and_streams_share_a_blocked_matrix(tb, gpu, per_column):
    """Runs in flight together on one matrix with blocked products, each against the run made alone.  A run stops
    within 1e-10 (L1) of the fixed point (sum-normalised), or where a step is below 1e-8 of iterates of sum at least
    1, so within 1e-8 * 0.85 / 0.15 of it; products of another run move it by far more."""
    import torch
    n = 70001
    m = tb.MatrixCSR().fill_cqmat_stochastic(n, n, 8, 0.5, 7, device=True)
    if not per_column:
        a = m.arrays()
        v = a["values"] * (0.5 + 0.5 * np.random.default_rng(1).random(a["values"].size))
        m = tb.MatrixCSR(n, n, v, a["rowptr"], a["colidx"])

    def blocked(k):
        out = torch.full((n,), -1.0, dtype=torch.float64, device="cuda")
        kw = dict(BLOCKED[k])
        eps = 1e-8 if kw["rule"] == "reference" else 1e-10
        m.page_rank_device(out, epsilon=eps, max_iteration=500, gather="blocked", **kw)
        return out.cpu()

    alone = [blocked(k) for k in range(len(BLOCKED))]
    torch.cuda.synchronize()
    seen, bad = [], []

    def work(t):
        with torch.cuda.stream(torch.cuda.Stream()):
            for r in range(8):
                k = (t + r) % len(BLOCKED)
                d = float((blocked(k) - alone[k]).abs().sum())
                seen.append(k)
                if not d <= (2e-10 if BLOCKED[k]["rule"] == "sumnorm" else 2e-7):
                    bad.append((t, BLOCKED[k], d))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert len(seen) == 32 and not bad, (len(seen), bad)
