"""Run memory kept with a matrix: runs of different sizes and kinds in turn,
and runs of several threads and streams on one matrix, equal runs on a fresh
matrix (whose memory nothing has used) bit for bit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N = 5003


def graph(tb):
    return tb.MatrixCSR().fill_cqmat_stochastic(N, N, 8, 0.5, 7)


def rank(m, torch, **kw):
    out = torch.full((N,), -1.0, dtype=torch.float64, device="cuda")
    rep = m.page_rank_device(out, epsilon=1e-10, max_iteration=300, gather="tiles", **kw)
    return out.cpu(), rep["iterations"]


KINDS = [{}, {"nodes": [3, 99]}, {"rule": "sumnorm", "precision": "f32"}, {"precision": "pattern"},
         {"rule": "sumnorm", "precision": "pattern_f32"}, {"rule": "sumnorm", "precision": "bf16"}]


def test_kinds_in_turn(tb, gpu):
    import torch
    fresh = [rank(graph(tb), torch, **k) for k in KINDS]
    m = graph(tb)
    w = torch.linspace(-1, 1, N, dtype=torch.float64, device="cuda")
    gt = torch.zeros(N, dtype=torch.float64, device="cuda")
    for _ in range(2):
        for k, (p, it) in zip(KINDS, fresh):
            q, jt = rank(m, torch, **k)
            assert torch.equal(p, q) and it == jt, k
            m.page_rank_adjoint(q.cuda(), w, grad_teleport=gt)
        p, it = m.page_rank(1e-10, 0.85, 300)
        assert np.array_equal(p, fresh[0][0].numpy()) and it == fresh[0][1]


def test_threads_and_streams_share_a_matrix(tb, gpu):
    import torch
    m = graph(tb)
    fresh = [rank(graph(tb), torch, **k) for k in KINDS]
    for k in KINDS:  # the lazily built mirrors exist before the threads start
        rank(m, torch, **k)
    torch.cuda.synchronize()
    bad = []

    def work(t):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for r in range(6):
                k = (t + r) % len(KINDS)
                p, it = rank(m, torch, **KINDS[k])
                if not (torch.equal(p, fresh[k][0]) and it == fresh[k][1]):
                    bad.append((t, KINDS[k]))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
