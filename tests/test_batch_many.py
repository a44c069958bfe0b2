"""Batches of few and of many small graphs, with and without a graph of several
sets: the sets of a graph come out the same, bit for bit, however many others
run beside it (their sums are over their own rows in one order), run after run
and whichever set ends last."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_many_small_graphs(tb, gpu, precision):
    import torch
    ns = [1, 2, 37, 64, 255, 256, 257, 700, 2049]
    gs = [tb.MatrixCSR().fill_cqmat_stochastic(n, n, min(n, 4), 0.4, 3 + n) for n in ns]
    kw = {"epsilon": 1e-9 if precision == "f64" else 1e-5, "max_iteration": 200, "rule": "sumnorm"}
    alone = []
    for n, g in zip(ns, gs):
        out, _, its = tb.PageRankBatch(precision).add_graph(g, [[n // 2]]).run(**kw)
        alone.append((out.cpu(), int(its[0])))
    big = tb.MatrixCSR().fill_cqmat_stochastic(1000, 1000, 6, 0.4, 9)
    sets = [[5 * k] for k in range(7)]
    for copies in (1, 3000):
        for group in (False, True):
            b = tb.PageRankBatch(precision)
            for k in range(copies):
                b.add_graph(gs[k % len(gs)], [[ns[k % len(gs)] // 2]])
            if group:
                b.add_graph(big, sets)
            for most in (200, 200, 3, 0):
                out, _, its = b.run(**{**kw, "max_iteration": most})
                torch.cuda.synchronize()
                off = b.layout()
                o = out.cpu()
                for k in range(copies):
                    p, it = alone[k % len(gs)]
                    assert its[k] == min(it, most), (copies, group, k, most)
                    assert most < 200 or torch.equal(o[off[k]:off[k + 1]], p), (copies, group, k)
