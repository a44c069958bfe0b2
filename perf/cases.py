"""What a user of this framework has it do on one GPU, as cases that can be timed.

Two families: products with a sparse (or dense) matrix in each of the five
formats, and PageRank in each of its forms -- the drop-in calls on host
vectors, the device-resident engine in every precision, many personalisation
vectors at once, and the differentiable call with its backward pass.  Every
case goes through the package's public entry points; the graphs come from the
package's own generators, which its tests and its benchmark use too.

    listed()             the cases, one per use
    draw(rng)            another case of the same ranges
    prepare(case, seed)  the matrix (mirrored in HBM) and the vectors
    run(state)           one pass
    work(case)           bytes and operations of one pass, at the least
    exact(case, seed)    the same results in 64 bits, from plain torch
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tbsla_amd as tb
from tbsla_amd.autograd import page_rank as differentiable_page_rank
from tbsla_amd.matrix import FORMATS

BETA = 0.85
VALUE_BYTES = {"f64": 8, "f32": 4, "bf16": 2, "pattern": 0, "pattern_f32": 0}


def listed():
    return [
        # the smallest product: the 10,000-row band matrix of the reference's own performance programs
        {"name": "csr_band_10k", "kind": "product", "format": "CSR", "matrix": "cdiag", "n": 10000, "c": 10, "q": 0.0,
         "grid": 1, "dtype": "f64"},
        # the benchmark product: one rank's block of a 4 x 4 distribution of a 2^24-row matrix
        {"name": "csr_block_2e24", "kind": "product", "format": "CSR", "matrix": "cqmat", "n": 1 << 24, "c": 16,
         "q": 0.1, "grid": 4, "dtype": "f64"},
        # an ordinary product with 32-bit values (a solver's inner product), rows padded to one length
        {"name": "ell_1m_f32", "kind": "product", "format": "ELL", "matrix": "cqmat", "n": 1000003, "c": 16, "q": 0.1,
         "grid": 1, "dtype": "f32"},
        # coordinate entries of an assembled matrix, accumulated into y
        {"name": "scoo_300k", "kind": "product", "format": "SCOO", "matrix": "cqmat", "n": 300007, "c": 12, "q": 0.2,
         "grid": 1, "dtype": "f64"},
        # a dense block at the largest size the format is meant for
        {"name": "dense_8192", "kind": "product", "format": "DENSE", "matrix": "cqmat", "n": 8192, "c": 64, "q": 0.5,
         "grid": 1, "dtype": "f64"},
        # the drop-in product of the reference's class: vectors on the host, copied both ways in the call
        {"name": "csr_host_vectors_1m", "kind": "host_product", "format": "CSR", "matrix": "cqmat", "n": 1000003,
         "c": 16, "q": 0.1, "grid": 1, "dtype": "f64"},
        # the drop-in PageRank call on a small graph (a service that ranks a subgraph per request)
        {"name": "pagerank_host_5k", "kind": "host_pagerank", "n": 5003, "c": 8, "q": 0.5, "nodes": 0,
         "epsilon": 1e-8},
        # a middling graph, FP64, to 1e-10 of the fixed point
        {"name": "pagerank_300k_f64", "kind": "pagerank", "n": 300007, "c": 16, "q": 0.2, "precision": "f64",
         "epsilon": 1e-10},
        # a large graph with 32-bit values, to the same accuracy
        {"name": "pagerank_5m_f32", "kind": "pagerank", "n": 5000011, "c": 8, "q": 0.5, "precision": "f32",
         "epsilon": 1e-10},
        # the benchmark graph of 2^24 nodes, FP64
        {"name": "pagerank_2e24_f64", "kind": "pagerank", "n": 1 << 24, "c": 8, "q": 0.5, "precision": "f64",
         "epsilon": 1e-10},
        # personalised PageRank of many users at once: graphs of uneven size with one node set each, and one
        # larger graph with 64 sets
        {"name": "batch_48_and_1m_x64", "kind": "batch", "graphs": 48, "lo": 10, "hi": 16, "c": 12, "big_n": 1 << 20,
         "big_c": 16, "sets": 64, "q": 0.3, "precision": "f32", "epsilon": 1e-5},
        # learning edge weights and a teleport distribution: the differentiable call and its backward pass
        {"name": "gradient_500k", "kind": "gradient", "n": 500009, "c": 16, "q": 0.2, "adjoint": "f32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["product", "product", "product", "host_product", "host_pagerank", "pagerank", "pagerank",
                       "batch", "gradient"])
    q = round(rng.uniform(0.02, 0.6), 3)
    if kind in ("product", "host_product"):
        fmt = rng.choice(["CSR", "CSR", "ELL", "SCOO", "COO", "DENSE"])
        if fmt == "DENSE":
            n, c, dtype = _log(rng, 300, 8192), 32, "f64"
        else:
            c = rng.randint(4, 32)
            n = _log(rng, 1000, min(1 << 22, 62000000 // c))
            dtype = "f64" if kind == "host_product" else rng.choice(["f64", "f64", "f32", "bf16"])
        return {"kind": kind, "format": fmt, "matrix": "cqmat", "n": n, "c": c, "q": q, "grid": 1, "dtype": dtype}
    if kind == "host_pagerank":
        return {"kind": kind, "n": _log(rng, 500, 60000), "c": rng.randint(4, 24), "q": q,
                "nodes": rng.choice([0, 0, 1, 5]), "epsilon": 1e-8}
    if kind == "pagerank":
        c = rng.randint(4, 20)
        return {"kind": kind, "n": _log(rng, 20000, min(1 << 24, 134000000 // c)), "c": c, "q": max(q, 0.1),
                "precision": rng.choice(["f64", "f64", "f32", "bf16", "pattern", "pattern_f32"]), "epsilon": 1e-10}
    if kind == "batch":
        precision = rng.choice(["f32", "f64"])
        return {"kind": kind, "graphs": rng.randint(4, 48), "lo": 9, "hi": rng.randint(12, 16),
                "c": rng.randint(6, 14), "big_n": _log(rng, 5000, 500000), "big_c": rng.randint(6, 16),
                "sets": rng.randint(2, 64), "q": max(q, 0.1), "precision": precision,
                "epsilon": 1e-5 if precision == "f32" else 1e-9}
    return {"kind": kind, "n": _log(rng, 1500, 500000), "c": rng.randint(4, 16), "q": max(q, 0.1),
            "adjoint": rng.choice(["f32", "f64"])}


def _seed32(seed):
    """A generator seed in [1, 2^31) from any whole number."""
    return int(seed) % ((1 << 31) - 1) + 1


def _uniform(n, seed, dtype=torch.float64):
    g = torch.Generator(device="cuda").manual_seed(_seed32(seed))
    return torch.rand(n, generator=g, dtype=dtype, device="cuda")


def _matrix(case, seed):
    m = FORMATS[case["format"]]()
    n, g = case["n"], case["grid"]
    if case["matrix"] == "cdiag":
        return m.fill_cdiag(n, n, case["c"], 0, 0, g, g)
    device = {} if case["format"] == "DENSE" else {"device": True}
    return m.fill_cqmat(n, n, case["c"], case["q"], _seed32(seed), 0, 0, g, g, value_seed=_seed32(seed), **device)


def _lengths(case):
    """(length of x, length of y) of a product."""
    n, g = case["n"], case["grid"]
    return (n // g, n // g)


def _graph(n, c, q, seed):
    return tb.MatrixCSR().fill_cqmat_stochastic(n, n, c, q, _seed32(seed), device=True)


def _nodes(case, seed):
    rng = np.random.default_rng(_seed32(seed))
    return rng.choice(case["n"], size=case["nodes"], replace=False).astype(np.int32)


def _batch_graphs(case, seed):
    """(n, c, graph seed, node sets) of each graph of a batch."""
    rng = np.random.default_rng(_seed32(seed))
    out = []
    for k in range(case["graphs"]):  # sizes spread over their logarithm
        n = int(2.0 ** (case["lo"] + (case["hi"] - case["lo"]) * (k + 0.5) / case["graphs"]))
        out.append((n, case["c"], seed + 1 + k, [[int(rng.integers(n))]]))
    big = case["big_n"]
    out.append((big, case["big_c"], seed, [[int(v)] for v in rng.integers(big, size=case["sets"])]))
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "product":
        m = s["matrix"] = _matrix(case, seed).prepare(case["dtype"])
        nx, ny = _lengths(case)
        vec = torch.float64 if case["dtype"] == "f64" else torch.float32
        s["x"] = _uniform(nx, seed, vec)
        s["y"] = torch.zeros(ny, dtype=vec, device="cuda")
        s["accumulates"] = m.NAME in ("COO", "SCOO", "DENSE")
    elif kind == "host_product":
        s["matrix"] = _matrix(case, seed).prepare("f64")
        s["x"] = np.random.default_rng(_seed32(seed)).random(_lengths(case)[0])
    elif kind == "host_pagerank":
        s["matrix"] = _graph(case["n"], case["c"], case["q"], seed).prepare("f64")
        s["nodes"] = _nodes(case, seed)
    elif kind == "pagerank":
        s["matrix"] = _graph(case["n"], case["c"], case["q"], seed).prepare("f64")
        s["out"] = torch.zeros(case["n"], dtype=torch.float64, device="cuda")
    elif kind == "batch":
        b = s["batch"] = tb.PageRankBatch(case["precision"])
        for n, c, gseed, sets in _batch_graphs(case, seed):
            b.add_graph(_graph(n, c, case["q"], gseed), sets)
        b.prepare()
        s["out"] = torch.zeros(int(b.layout()[-1]), dtype=torch.float64, device="cuda")
    else:
        m = s["matrix"] = _graph(case["n"], case["c"], case["q"], seed).prepare("f64")
        s["values"] = torch.from_numpy(m.arrays()["values"]).cuda().requires_grad_(True)
        t = _uniform(case["n"], seed) + 0.5
        s["teleport"] = (t / t.sum()).requires_grad_(True)
        s["w"] = _uniform(case["n"], seed + 1) - 0.5
    return s


def run(s):
    case, kind = s["case"], s["kind"]
    if kind == "product":
        if s["accumulates"]:  # y += A x: a fresh result starts from zero
            s["y"].zero_()
        return s["matrix"].Ax_device(s["x"], s["y"], value_dtype=case["dtype"])
    if kind == "host_product":
        return s["matrix"].spmv(s["x"])
    if kind == "host_pagerank":
        m = s["matrix"]
        if case["nodes"]:
            p, its = m.personalized_page_rank(case["epsilon"], BETA, 500, s["nodes"])
        else:
            p, its = m.page_rank(case["epsilon"], BETA, 500)
        return {"rank": p, "iterations": its}
    if kind == "pagerank":
        rep = s["matrix"].page_rank_device(s["out"], epsilon=case["epsilon"], beta=BETA, max_iteration=500,
                                           precision=case["precision"], rule="sumnorm")
        return {"rank": s["out"], "iterations": rep["iterations"]}
    if kind == "batch":
        out, _, its = s["batch"].run(out=s["out"], epsilon=case["epsilon"], beta=BETA, max_iteration=500,
                                     rule="sumnorm")
        return {"ranks": out, "iterations": its}
    s["values"].grad = s["teleport"].grad = None
    p = differentiable_page_rank(s["matrix"], s["values"], s["teleport"], beta=BETA, epsilon=1e-13,
                                 adjoint_precision=case["adjoint"],
                                 adjoint_epsilon=1e-7 if case["adjoint"] == "f32" else 1e-12)
    (s["w"] * p).sum().backward()
    return {"rank": p.detach(), "d_values": s["values"].grad, "d_teleport": s["teleport"].grad}


def _entries(case):
    """Stored entries of a product's matrix (about)."""
    nx, ny = _lengths(case)
    if case["format"] == "DENSE":
        return nx * ny
    if case["matrix"] == "cdiag":
        return 2 * ny
    # a block on the diagonal of a grid keeps the band and 1/grid of the rewired entries
    keep = (1 - case["q"]) + case["q"] / case["grid"]
    return int(ny * case["c"] * (keep if case["format"] != "ELL" else 1))


def work(case):
    """Each input once and each result once.  PageRank reads the graph again
    in every iteration; how many it takes depends on the graph, and they are
    not counted here."""
    kind = case["kind"]
    if kind in ("product", "host_product"):
        e, (nx, ny) = _entries(case), _lengths(case)
        vb = VALUE_BYTES[case["dtype"]]
        xb = 8 if case["dtype"] == "f64" else 4
        index = {"CSR": 4 * e + 4 * ny, "ELL": 4 * e, "SCOO": 8 * e, "COO": 8 * e, "DENSE": 0}[case["format"]]
        return {"bytes": e * vb + index + xb * (nx + ny), "flops": 2 * e}
    n = case.get("n", 0)
    e = n * case.get("c", 0)
    if kind in ("host_pagerank", "pagerank"):
        vb = VALUE_BYTES[case.get("precision", "f64")]
        return {"bytes": e * (4 + vb) + 4 * n + 8 * n, "flops": 2 * e}
    if kind == "batch":
        vb = VALUE_BYTES[case["precision"]]
        mean = (2.0 ** case["hi"] - 2.0 ** case["lo"]) / (math.log(2) * max(1, case["hi"] - case["lo"]))
        small, big = int(case["graphs"] * mean), case["big_n"]
        return {"bytes": (small * case["c"] + big * case["big_c"]) * (4 + vb) + 8 * (small + big * case["sets"]),
                "flops": 2 * (small * case["c"] + big * case["big_c"] * case["sets"])}
    return {"bytes": e * (4 + 8 + 8) + 4 * n + 8 * n * 4, "flops": 6 * e}


# ---- the same results in 64 bits, from plain torch -------------------------


def _triples(m):
    """(rows, columns, values) of a matrix's stored entries, local to its block, on the GPU."""
    a, i = m.arrays(), m.info()
    f_row, f_col = i["f_row"], i["f_col"]
    v = torch.from_numpy(a["values"]).cuda()
    if m.NAME == "CSR":
        ptr = torch.from_numpy(a["rowptr"]).cuda().long()
        r = torch.repeat_interleave(torch.arange(ptr.numel() - 1, device="cuda"), ptr[1:] - ptr[:-1])
        return r, torch.from_numpy(a["colidx"]).cuda().long()[: r.numel()] - f_col, v[: r.numel()]
    if m.NAME == "ELL":
        k = i["max_col"]
        r = torch.arange(v.numel(), device="cuda") // k
        return r, (torch.from_numpy(a["columns"]).cuda().long() - f_col).clamp_(min=0), v
    if m.NAME == "DENSE":
        at = torch.arange(v.numel(), device="cuda")
        return at // i["ln_col"], at % i["ln_col"], v
    r, c = (torch.from_numpy(a[k]).cuda().long() for k in ("row", "col"))
    return (r - f_row, c - f_col, v) if m.NAME == "SCOO" else (r, c, v)


def _fixed_point(r, c, v, teleport, most=1500, enough=1e-15):
    """The sum-normalised fixed point of x = beta A x + (1 - beta) (1^T x) teleport, for each column of teleport."""
    x = torch.full_like(teleport, 1.0 / teleport.shape[0])
    some = max(1, (1 << 28) // teleport[0].numel())  # entries at a time
    best = math.inf
    for _ in range(most):
        y = torch.zeros_like(x)
        for k in range(0, r.numel(), some):
            part = v[k:k + some].reshape(-1, *[1] * (x.dim() - 1)) * x[c[k:k + some]]
            y.index_add_(0, r[k:k + some], part)
        y.mul_(BETA).add_(teleport * ((1 - BETA) * x.sum(0)))
        y /= y.sum(0)
        step = float((y - x).abs().sum(0).max())
        x = y
        if step < enough or (step < 1e-13 and step >= best):
            break
        best = min(best, step)
    return x


def _one_hot(n, nodes):
    t = torch.zeros(n, dtype=torch.float64, device="cuda")
    t[torch.as_tensor(np.asarray(nodes), device="cuda").long()] = 1.0 / len(nodes)
    return t


def exact(case, seed):
    kind = case["kind"]
    if kind in ("product", "host_product"):
        s = prepare(case, seed)
        r, c, v = _triples(s["matrix"])
        x = torch.as_tensor(s["x"]).cuda().double()
        return torch.zeros(_lengths(case)[1], dtype=torch.float64, device="cuda").index_add_(0, r, v * x[c])
    if kind in ("host_pagerank", "pagerank"):
        n = case["n"]
        r, c, v = _triples(_graph(n, case["c"], case["q"], seed))
        uniform = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
        t = _one_hot(n, _nodes(case, seed)) if case.get("nodes") else uniform
        return {"rank": _fixed_point(r, c, v, t), "iterations": None}
    if kind == "batch":
        parts = []
        for n, c, gseed, sets in _batch_graphs(case, seed):
            r, cc, v = _triples(_graph(n, c, case["q"], gseed))
            t = torch.stack([_one_hot(n, nodes) for nodes in sets], dim=1)
            parts.append(_fixed_point(r, cc, v, t, enough=1e-12).t().reshape(-1))
        return {"ranks": torch.cat(parts), "iterations": None}
    s = prepare(case, seed)
    n = case["n"]
    r, c, v = _triples(s["matrix"])
    t, w = s["teleport"].detach(), s["w"]
    p = _fixed_point(r, c, v, t)
    # gradient through p = M p / (1^T M p), M = beta A + (1 - beta) t 1^T
    total = BETA * (v * p[c]).sum() + (1 - BETA) * t.sum() * p.sum()
    lam = w.clone()
    for _ in range(400):
        g = (lam - torch.dot(p, lam)) / total
        new = torch.zeros_like(lam).index_add_(0, c, v * g[r]).mul_(BETA).add_((1 - BETA) * torch.dot(t, g)).add_(w)
        step = float((new - lam).abs().sum() / new.abs().sum())
        lam = new
        if step < 1e-15:
            break
    g = (lam - torch.dot(p, lam)) / total
    return {"rank": p, "d_values": BETA * g[r] * p[c], "d_teleport": (1 - BETA) * p.sum() * g}
