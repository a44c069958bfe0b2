"""Benchmark: SpMV GB/s as % of HBM peak, and PageRank time to 1e-10 L1.

Workload (one GPU): rank (0,0)'s block of a 4x4 2D distribution of
fill_cqmat(2^24, 2^24, c=16, q=0.1, seed 42) -- 4,194,304 x 4,194,304,
62,075,592 entries -- with values 1 - u01(42, i) and x_j = u01(1, j).
A step is one FP64 CSR SpMV of that block with the inputs resident in HBM.
The W warm-up steps follow about 50 ms of untimed steps that bring the GPU's
clocks up after the host work before the leg; the K timed steps follow.

CSR matrices are generated on the GPU (fill_cqmat(..., device=True)), which
gives the host generators' arrays; the other formats are generated on the
host.

Extra fields:
  formats        ELL / SCOO / COO / DENSE on the same block
  cpu_baseline   the reference's own MatrixCSR::Ax and spmv() (compiled from
                 its sources) on the host cores, best and median of 10, and
                 the bit-exact check of the GPU y; its Matrix::page_rank on
                 the PageRank graph, per iteration and to 1e-10.  Each is
                 timed with the reference's thread binding (OMP_PLACES=cores
                 OMP_PROC_BIND=close) and with unbound threads; the faster
                 setting is the baseline, both are reported
  pagerank       fill_cqmat_stochastic(2^24, 2^24, 8, 0.5, 7) in FP64, FP32 and
                 BF16 value storage, value-free FP64 and value-free FP32, each
                 stopped by the sum-normalised bound (median of three runs
                 each), against the FP64 fixed point p* computed on the host
                 by the oracle (whose digest is the reference's own vector)
  batch          256 personalised graphs (n log-uniform in [2^10, 2^18]) plus
                 a 2^22-node graph with 64 one-hot teleport sets, one hipGraph
  adjoint        gradient of sum w_i p_i on fill_cqmat_stochastic(2^20, 2^20,
                 16, 0.2, 3), FP32 and FP64 transposed products

    python bench.py [--steps K] [--warmup W] [--no-pagerank] [--no-cpu]
                    [--no-formats] [--no-batch] [--no-adjoint]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
METRIC = "SpMV GB/s as % of HBM peak; PageRank s-to-1e-10 L1 (mixed vs FP64 GPU)"
N = 1 << 24


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


SETTLE_S = 0.05  # device time of untimed calls that bring the clocks up before the warm-up steps


def time_kernel(torch, fn, steps, warmup, batches=1):
    """Average device time per call of fn() over `steps` calls, measured with
    HIP events on torch's current stream (the stream the kernels run on).
    With batches > 1 the calls are split into that many consecutive groups
    with an event between groups, and the per-call time of each group is
    returned as well: (mean over all steps, [per-group means]).

    Before the `warmup` calls, about SETTLE_S seconds of untimed calls: after
    the host work that precedes a leg the GPU is idle, and the first calls
    after an idle gap of 0.5-2 s run 7-10% slower (measured on the CSR block:
    5050-5200 GB/s in the first four calls, 5600-5650 after), which a few
    warm-up calls of ~0.15 ms do not cover."""
    for _ in range(4):
        fn()
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(4):
        fn()
    torch.cuda.synchronize()
    per = max((time.perf_counter() - t) / 4, 1e-5)
    for _ in range(min(2000, int(SETTLE_S / per))):
        fn()
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    s = torch.cuda.current_stream()
    nb = max(1, min(batches, steps))
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(nb + 1)]
    sizes = [steps // nb + (1 if b < steps % nb else 0) for b in range(nb)]
    ev[0].record(s)
    for b in range(nb):
        for _ in range(sizes[b]):
            fn()
        ev[b + 1].record(s)
    torch.cuda.synchronize()
    total = ev[0].elapsed_time(ev[nb]) / steps
    if batches == 1:
        return total
    return total, [ev[b].elapsed_time(ev[b + 1]) / sizes[b] for b in range(nb)]


def pmc_traffic(name):
    """HBM bytes per launch from the committed rocprofv3 counter summary, if any."""
    path = os.path.join(ROOT, "profiles", f"{name}_pmc.txt")
    if not os.path.exists(path):
        return None
    for line in open(path):
        if line.startswith("traffic_bytes_per_launch"):
            return float(line.split("=")[1])
    return None


def _dump_csr(d, arrays, **meta):
    """Raw CSR arrays and their sizes for the CPU-baseline child process."""
    for k in ("values", "rowptr", "colidx"):
        arrays[k].tofile(os.path.join(d, f"{k}.bin"))
    meta.update({"n_values": int(arrays["values"].size), "n_rowptr": int(arrays["rowptr"].size),
                 "n_colidx": int(arrays["colidx"].size)})
    with open(os.path.join(d, "meta.json"), "w") as f:
        json.dump(meta, f)


def _cpu_child(task, d, bind=True):
    """Run oracle/cpu_baseline.py in a child process with the OpenMP
    environment of a reference run: all the host threads this job may use,
    and with `bind` OMP_PLACES=cores OMP_PROC_BIND=close (as the reference's
    machine files set it), else the threads left unbound."""
    import subprocess
    from oracle.cpu_baseline import host_cores, omp_env
    cores = host_cores()
    r = subprocess.run([sys.executable, "-m", "oracle.cpu_baseline", task, d], cwd=ROOT,
                       env=omp_env(cores["threads"], bind), capture_output=True, text=True, timeout=900)
    if r.returncode != 0:
        raise RuntimeError(f"cpu_baseline {task} failed: {r.stderr[-2000:]}")
    res = json.loads(r.stdout.strip().splitlines()[-1])
    res["cores"] = cores
    return res


OMP_BOUND = "OMP_PLACES=cores OMP_PROC_BIND=close"
OMP_FREE = "OMP_PROC_BIND=false (threads placed by the OS)"


def cpu_baseline(tb_csr, x, y_gpu, bytes_alg):
    """The reference's own CSR Ax and spmv() (oracle/_ref, compiled from its
    sources, -O3 -fopenmp) on the same block, timed on the host cores in a
    child process, once with the reference's thread binding and once with
    unbound threads (the faster is the baseline); its result is compared
    with the GPU product (bit-exact)."""
    import hashlib
    import shutil
    import tempfile
    from oracle.oracle import Reference
    if not Reference.available():
        return None
    info = tb_csr.info()
    d = tempfile.mkdtemp(prefix="tbsla_cpu_")
    try:
        _dump_csr(d, tb_csr.arrays(), n_row=info["ln_row"], n_col=info["ln_col"])
        x.tofile(os.path.join(d, "x.bin"))
        runs = {OMP_BOUND: _cpu_child("spmv", d, bind=True), OMP_FREE: _cpu_child("spmv", d, bind=False)}
    finally:
        shutil.rmtree(d, ignore_errors=True)
    gbs = lambda t: round(bytes_alg / t / 1e9, 2)  # noqa: E731
    setting = min(runs, key=lambda k: runs[k]["Ax"]["median_s"])
    res = runs[setting]
    ax, sp, cores = res["Ax"], res["spmv_api"], res["cores"]
    return {"value": gbs(ax["median_s"]), "unit": "GB/s", "cores": cores["threads"], "kind": "reference",
            "sample": f"MatrixCSR::Ax on the full block, 1 warm-up + {ax['runs']} timed runs (median; best "
                      f"{ax['best_s'] * 1e3:.1f} ms, median {ax['median_s'] * 1e3:.1f} ms), reference sources "
                      f"g++ -O3 -fopenmp, {cores['threads']} threads, {setting} (the faster of the two settings)",
            "host": cores,
            "Ax": {"best_gbs": gbs(ax["best_s"]), "median_gbs": gbs(ax["median_s"]),
                   "best_ms": round(ax["best_s"] * 1e3, 3), "median_ms": round(ax["median_s"] * 1e3, 3)},
            "spmv_api": {"note": "spmv() returns a zeroed n_row-length vector (MatrixCSR.cpp:123-127)",
                         "best_ms": round(sp["best_s"] * 1e3, 3), "median_ms": round(sp["median_s"] * 1e3, 3),
                         "median_gbs": gbs(sp["median_s"])},
            "omp_settings": {k: {"Ax_median_ms": round(v["Ax"]["median_s"] * 1e3, 3),
                                 "Ax_best_ms": round(v["Ax"]["best_s"] * 1e3, 3),
                                 "spmv_api_median_ms": round(v["spmv_api"]["median_s"] * 1e3, 3)}
                             for k, v in runs.items()},
            "gpu_y_bit_exact_vs_reference": all(v["y_sha256"] == hashlib.sha256(y_gpu.tobytes()).hexdigest()
                                                for v in runs.values())}


def copy_calibration():
    """Five copies of 2^27 doubles: 1 GiB read and 1 GiB written per launch."""
    import torch
    src = torch.ones(1 << 27, dtype=torch.float64, device="cuda:0")
    dst = torch.empty_like(src)
    ms = time_kernel(torch, lambda: dst.copy_(src), 5, 1)
    log(f"copy of {src.numel() * 8} bytes: {ms * 1e3:.1f} us, {2 * src.numel() * 8 / ms / 1e6:.0f} GB/s")


def leg_formats(torch, tb, dev, steps):
    fm = {}
    for fmt in ["ELL", "SCOO", "COO"]:
        m = tb.FORMATS[fmt]().fill_cqmat(N, N, 16, 0.1, 42, 0, 0, 4, 4, value_seed=42)
        mi2 = m.mirror_info("f64")
        nx = N if fmt == "COO" else m.get_ln_col()
        xx = torch.from_numpy(tb.u01_array(1, 0, nx)).to(dev)
        yy = torch.zeros(m.get_n_row(), dtype=torch.float64, device=dev)
        ms2 = time_kernel(torch, lambda: m.Ax_device(xx, yy), max(10, steps // 4), 3)
        fm[fmt] = {"us": round(ms2 * 1e3, 1), "gbs": round(mi2["algorithmic_bytes"] / ms2 / 1e6, 1),
                   "bytes": mi2["algorithmic_bytes"]}
        if fmt in ("SCOO", "COO"):
            # the kernel reads the compressed-row mirror, not the format's
            # arrays: 12 B per entry, 8 B per row segment, x once, y read and
            # written.  Those are the bytes it must move, so they are the
            # primary figure; the format's own bytes are kept beside it.
            mb = mi2["entries"] * 12 + mi2["rows"] * 8 + 8 * mi2["x_need"] + 16 * (mi2["y_hi"] - mi2["y_lo"])
            fm[fmt] = {"us": fm[fmt]["us"], "gbs": round(mb / ms2 / 1e6, 1), "bytes": mb,
                       "bytes_model": "compressed-row mirror read by the kernel",
                       "format_bytes": mi2["algorithmic_bytes"],
                       "format_bytes_gbs": round(mi2["algorithmic_bytes"] / ms2 / 1e6, 1)}
        fm[fmt]["pct_hbm_peak"] = round(fm[fmt]["gbs"] / HBM_PEAK_GBS * 100, 2)
        log(f"{fmt} {ms2 * 1e3:.1f} us {fm[fmt]['gbs']} GB/s")
        del m, xx, yy
        torch.cuda.empty_cache()
    m = tb.MatrixDENSE().fill_cqmat(32768, 32768, 16, 0.1, 42, 0, 0, 4, 4, value_seed=42)
    mi2 = m.mirror_info("f64")
    xx = torch.from_numpy(tb.u01_array(1, 0, 8192)).to(dev)
    yy = torch.zeros(32768, dtype=torch.float64, device=dev)
    ms2 = time_kernel(torch, lambda: m.Ax_device(xx, yy), 20, 3)
    fm["DENSE"] = {"us": round(ms2 * 1e3, 1), "gbs": round(mi2["algorithmic_bytes"] / ms2 / 1e6, 1),
                   "bytes": mi2["algorithmic_bytes"]}
    log(f"DENSE {ms2 * 1e3:.1f} us {fm['DENSE']['gbs']} GB/s")
    return fm


PSTAR_ITERATIONS = 48   # the reference iteration is in its limit 2-cycle from ~40 iterations on
REF_RULE_ITERATIONS = 26  # the drop-in (reference-rule) runs, timed per iteration
CPU_PR_SAMPLE = 5       # reference page_rank iterations timed on the host


def leg_pagerank(torch, tb, dev, cpu=True):
    """Every precision to the sum-normalised 1e-10 bound (median of three
    timed runs each), then the FP64 fixed point p* on the host (the oracle's
    restatement of the reference iteration, 48 iterations; its SHA-256 is
    checked against the reference's own vector) and the reference CPU
    page_rank timed on a bounded sample of iterations."""
    import hashlib
    import shutil
    import tempfile
    log("generating the PageRank graph")
    g = tb.MatrixCSR().fill_cqmat_stochastic(N, N, 8, 0.5, 7, device=True)
    n = g.get_n_col()
    pr, outs = {}, {}
    for prec in ["f64", "f32", "bf16", "pattern", "pattern_f32"]:
        o = torch.zeros(n, dtype=torch.float64, device=dev)
        g.page_rank_device(o, epsilon=1e-10, max_iteration=300, precision=prec, rule="sumnorm")  # warm
        # the median of three timed runs (one run varies by 1-2%)
        reps = [g.page_rank_device(o, epsilon=1e-10, max_iteration=300, precision=prec, rule="sumnorm")
                for _ in range(3)]
        rep = sorted(reps, key=lambda r: r["seconds"])[1]
        outs[prec] = o
        pr[prec] = {"seconds": round(rep["seconds"], 6), "runs": 3, "run_seconds": [round(r["seconds"], 6) for r in reps],
                    "iterations": rep["iterations"], "anchors": rep["anchors"]}
        log(f"pagerank {prec}: {rep['seconds'] * 1e3:.2f} ms, {rep['iterations']} it, {rep['anchors']} anchors")
    base = pr["f64"]["seconds"]
    for prec in pr:
        pr[prec]["speedup_vs_fp64"] = round(base / pr[prec]["seconds"], 3)
    # the value-free FP32 scheme against the value-free FP64 path as well
    pr["pattern_f32"]["speedup_vs_fp64_pattern"] = round(pr["pattern"]["seconds"] / pr["pattern_f32"]["seconds"], 3)
    # the drop-in page_rank() path: the reference's stopping rule (which
    # never fires at this size: 2-cycle at 2.5e-9), a fixed number of
    # iterations, with propagation-blocked products (the default) and with
    # fixed-order tiles (gather="tiles", the reference's summation order)
    ref_rule = {}
    for gather in ("auto", "tiles"):
        o = torch.zeros(n, dtype=torch.float64, device=dev)
        g.page_rank_device(o, epsilon=0.0, max_iteration=4, precision="f64", rule="reference", gather=gather)  # warm
        rep = g.page_rank_device(o, epsilon=0.0, max_iteration=REF_RULE_ITERATIONS, precision="f64", rule="reference",
                                 gather=gather)
        ref_rule["propagation_blocked" if gather == "auto" else "tiles"] = {
            "iterations": rep["iterations"], "seconds": round(rep["seconds"], 6),
            "ms_per_iteration": round(rep["seconds"] / rep["iterations"] * 1e3, 3)}
        log(f"pagerank reference rule ({gather}): {rep['seconds'] / rep['iterations'] * 1e3:.3f} ms per iteration")
        del o
    # the GPU's own FP64 limit: the reference iteration on fixed-order tiles
    lim = torch.zeros(n, dtype=torch.float64, device=dev)
    g.page_rank_device(lim, epsilon=0.0, max_iteration=PSTAR_ITERATIONS, precision="f64", rule="reference",
                       gather="tiles")
    out = {"graph": "fill_cqmat_stochastic(2^24,2^24,8,0.5,7), beta 0.85",
           "stop": "sum-normalised L1 bound <= 1e-10*(1-beta)/beta", "variants": pr,
           "reference_rule": ref_rule}
    if not cpu:  # (--no-cpu: no host legs; the GPU's own FP64 limit is the reference point)
        for prec, o in outs.items():
            pr[prec]["l1_vs_gpu_fp64_limit"] = float((o - lim).abs().sum().item())
        return out
    log("FP64 fixed point on the host (oracle) and the reference CPU page_rank")
    d = tempfile.mkdtemp(prefix="tbsla_pr_")
    try:
        _dump_csr(d, g.arrays(), n=n, beta=0.85, pstar_iterations=PSTAR_ITERATIONS, sample_iterations=CPU_PR_SAMPLE)
        res = _cpu_child("pagerank", d, bind=True)
        pstar = np.fromfile(os.path.join(d, "pstar.bin"), dtype=np.float64)
        free = _cpu_child("pagerank-time", d, bind=False) if "reference" in res else {}
    finally:
        shutil.rmtree(d, ignore_errors=True)
    with open(os.path.join(ROOT, "tests", "golden", "digests.json")) as f:
        fix = json.load(f)["pagerank_cfg3"]
    ps = torch.from_numpy(pstar).to(dev)
    out["pstar"] = {"source": f"oracle restatement of Matrix.cpp:13-61, {PSTAR_ITERATIONS} iterations, host",
                    "equals_reference_vector": res["pstar"]["sha256"] == fix[f"it{PSTAR_ITERATIONS}"]["sha256"]
                    and hashlib.sha256(pstar.tobytes()).hexdigest() == res["pstar"]["sha256"],
                    "host_seconds": round(res["pstar"]["seconds"], 2),
                    "gpu_fp64_limit_l1": float((lim - ps).abs().sum().item())}
    for prec, o in outs.items():
        pr[prec]["l1_vs_oracle_pstar"] = float((o - ps).abs().sum().item())
        log(f"pagerank {prec}: L1 vs oracle p* {pr[prec]['l1_vs_oracle_pstar']:.2e}")
    if "reference" in res:
        it_f64 = pr["f64"]["iterations"]
        settings = {OMP_BOUND: res["reference"]}
        if "reference" in free:
            settings[OMP_FREE] = free["reference"]
        setting = min(settings, key=lambda k: settings[k]["seconds_per_iteration"])
        spi = settings[setting]["seconds_per_iteration"]
        out["cpu_baseline"] = {
            "kind": "reference", "cores": res["cores"]["threads"],
            "sample": f"Matrix::page_rank (reference sources, -O3 -fopenmp) for {res['reference']['iterations']} "
                      f"iterations on the same graph, {res['cores']['threads']} threads, {setting} "
                      "(the faster of the two settings)",
            "seconds_per_iteration": round(spi, 4),
            "omp_settings": {k: round(v["seconds_per_iteration"], 4) for k, v in settings.items()},
            "iterations_to_1e-10": it_f64,
            "seconds_to_1e-10": round(spi * it_f64, 3),
            "note": "the reference's own stopping quantity never falls below ~2e-9 at this size (2-cycle); "
                    "the FP64 iteration count of the sum-normalised bound is used for both",
            "gpu_fp64_speedup": round(spi * it_f64 / pr["f64"]["seconds"], 1)}
    del outs, ps, lim
    return out


def leg_batch(torch, tb, dev):
    log("generating the personalised batch (256 graphs + 2^22 x 64)")
    t = time.time()
    spec = tb.personalised_workload()
    mats = [tb.MatrixCSR().fill_cqmat_stochastic(n, n, c, q, s, device=True) for (n, c, q, s, _) in spec]
    log(f"generated in {time.time() - t:.1f}s")
    res = {}
    outs = {}
    for prec, eps in (("f32", 1e-6), ("f64", 1e-10)):
        b = tb.PageRankBatch(prec)
        for m, sp in zip(mats, spec):
            b.add_graph(m, sp[4])
        t = time.time()
        b.prepare()
        prep = time.time() - t
        out, rep, its = b.run(epsilon=eps, rule="sumnorm", max_iteration=1000, check_every=16)
        out2, rep2, _ = b.run(out=out, epsilon=eps, rule="sumnorm", max_iteration=1000, check_every=16)
        # a second batch of the same graphs and sets: the autotuner's cache
        # gives it the shape with no trial iterations
        b2 = tb.PageRankBatch(prec)
        for m, sp in zip(mats, spec):
            b2.add_graph(m, sp[4])
        _, rep3, _ = b2.run(out=out, epsilon=eps, rule="sumnorm", max_iteration=1000, check_every=16)
        del b2
        res[prec] = {"seconds": round(rep2["seconds"], 6), "iterations_max": int(rep2["iterations"]),
                     "iterations_total": int(its.sum()), "stop": f"sum-normalised bound <= {eps}*(1-beta)/beta",
                     "bytes_per_iteration": rep2["bytes_per_iteration"],
                     "autotuned": rep["config"],
                     "first_run": {"seconds": round(rep["seconds"], 6), "tune_seconds": round(rep["tune_seconds"], 4),
                                   "tune_iterations": rep["tune_iterations"],
                                   # what the trials cost beyond the iterations they ran: the first
                                   # run against the later runs of the same batch in the chosen shape
                                   "tune_overhead_seconds": round(rep["seconds"] - min(rep2["seconds"], rep3["seconds"]), 5),
                                   "tune_overhead_fraction": round((rep["seconds"] - min(rep2["seconds"], rep3["seconds"]))
                                                                   / rep["seconds"], 4)},
                     "second_batch": {"seconds": round(rep3["seconds"], 6), "tune_cached": rep3["tune_cached"],
                                      "tune_seconds": round(rep3["tune_seconds"], 5),
                                      "tune_iterations": rep3["tune_iterations"]},
                     "prepare_seconds": round(prep, 2)}
        outs[prec] = (b.layout(), out2.cpu().numpy())
        log(f"batch {prec}: {rep2['seconds'] * 1e3:.1f} ms, max {rep2['iterations']} it, config {rep['config']}")
        del b, out, out2
        torch.cuda.empty_cache()
    off, p32 = outs["f32"]
    _, p64 = outs["f64"]
    l1 = [float(np.abs(p32[off[k]:off[k + 1]] - p64[off[k]:off[k + 1]]).sum()) for k in range(len(off) - 1)]
    res["f32"]["max_l1_vs_f64_batch"] = max(l1)
    # how the reference runs it: one personalised call per teleport set (sampled)
    big, (n, c, q, s, sets) = mats[-1], spec[-1]
    o = torch.zeros(n, dtype=torch.float64, device=dev)
    secs = []
    for nodes in sets[:4]:
        rep = big.page_rank_device(o, epsilon=1e-10, max_iteration=1000, precision="f64", rule="sumnorm", nodes=nodes)
        secs.append(rep["seconds"])
    res["single_call_per_set_f64"] = {"sample": "4 of the 64 sets of the 2^22 graph, FP64 single-graph engine",
                                      "seconds_per_set": round(float(np.mean(secs)), 6)}
    return {"workload": "256 x fill_cqmat_stochastic(n_g,n_g,12,0.3,1000+g), n_g log-uniform [2^10,2^18], one "
                        "one-hot set each; fill_cqmat_stochastic(2^22,2^22,16,0.3,1256) with 64 one-hot sets",
            "n_sets": len(off) - 1, "variants": res}


def leg_adjoint(torch, tb, dev):
    log("generating the adjoint graph")
    n = 1 << 20
    g = tb.MatrixCSR().fill_cqmat_stochastic(n, n, 16, 0.2, 3, device=True)
    p = torch.empty(n, dtype=torch.float64, device=dev)
    fwd = g.page_rank_device(p, epsilon=1e-15, max_iteration=400, rule="sumnorm")
    w = torch.from_numpy(tb.normal_array(3, n)).to(dev)
    ne = g.n_entries()
    res = {"forward_seconds": round(fwd["seconds"], 6), "forward_iterations": fwd["iterations"]}
    grads = {}
    for prec, eps in (("f32", 1e-7), ("f64", 1e-13)):
        gv = torch.zeros(ne, dtype=torch.float64, device=dev)
        gt = torch.zeros(n, dtype=torch.float64, device=dev)
        g.page_rank_adjoint(p, w, gv, gt, precision=prec, epsilon=eps)  # warm (builds A^T)
        rep = g.page_rank_adjoint(p, w, gv, gt, precision=prec, epsilon=eps)
        res[prec] = {"seconds": round(rep["seconds"], 6), "iterations": rep["iterations"],
                     "last_change": rep["last_change"]}
        grads[prec] = (gv, gt)
        log(f"adjoint {prec}: {rep['seconds'] * 1e3:.2f} ms, {rep['iterations']} it")
    (a, b), (c, d) = grads["f32"], grads["f64"]
    res["f32"]["rel_err_edge_grad_vs_f64"] = float(((a - c).abs().max() / c.abs().max()).item())
    res["f32"]["rel_err_teleport_grad_vs_f64"] = float(((b - d).abs().max() / d.abs().max()).item())
    return {"graph": "fill_cqmat_stochastic(2^20,2^20,16,0.2,3), beta 0.85, w ~ N(0,1) seed 3", **res}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--no-pagerank", action="store_true")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-formats", action="store_true")
    ap.add_argument("--no-batch", action="store_true")
    ap.add_argument("--no-adjoint", action="store_true")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run a plain 1 GiB device copy (the reference kernel for the "
                         "FETCH_SIZE / WRITE_SIZE counter scale)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU's block: there is no multi-GPU path (sharding over the "
              "2D block grid is not built); run with --gpus 1", file=sys.stderr)
        sys.exit(2)
    if args.copy_calibration:
        copy_calibration()
        return

    import torch
    import tbsla_amd as tb

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    log("generating the CSR block")
    t = time.time()
    csr = tb.MatrixCSR().fill_cqmat(N, N, 16, 0.1, 42, 0, 0, 4, 4, value_seed=42, device=True)
    log(f"generated in {time.time() - t:.1f}s")
    info = csr.info()
    x_host = tb.u01_array(1, 0, info["ln_col"])
    x = torch.from_numpy(x_host).to(dev)
    y = torch.zeros(info["ln_row"], dtype=torch.float64, device=dev)
    csr.prepare("f64")
    mi = csr.mirror_info("f64")
    ms, per_batch = time_kernel(torch, lambda: csr.Ax_device(x, y), args.steps, args.warmup, batches=5)
    gbs = mi["algorithmic_bytes"] / (ms * 1e-3) / 1e9
    batch_gbs = sorted(mi["algorithmic_bytes"] / (b * 1e-3) / 1e9 for b in per_batch)
    log(f"CSR {ms * 1e3:.1f} us/launch {gbs:.0f} GB/s ({100 * gbs / HBM_PEAK_GBS:.1f}% of peak)")
    # the C-ABI host-vector path (x and y cross PCIe inside the call)
    t = time.perf_counter()
    for _ in range(5):
        csr.spmv(x_host)
    host_ms = (time.perf_counter() - t) / 5 * 1e3

    out = {"metric": METRIC, "value": round(gbs, 2), "unit": "GB/s", "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "ms_per_step": round(ms, 5), "higher_is_better": True, "scaling": "weak",
           "vs_baseline": None, "dtype": "f64", "data": "synthetic",
           "config": {"workload": "CSR SpMV, block (0,0) of a 4x4 grid over fill_cqmat(2^24,2^24,16,0.1,42)",
                      "n_row": info["ln_row"], "n_col": info["ln_col"], "nnz": info["n_values"],
                      "values": "1-u01(42,i)", "x": "u01(1,j)", "pct_hbm_peak": round(100 * gbs / HBM_PEAK_GBS, 2),
                      "host_vector_spmv_ms": round(host_ms, 2)},
           "roofline": {"bound": "hbm", "achieved": round(gbs, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                        "frac": round(gbs / HBM_PEAK_GBS, 4), "traffic": pmc_traffic("csr_tile_kernel_cqmat2^24_block"),
                        "kernel": "csr_tile_kernel<double,double,double>",
                        "algorithmic_bytes_per_launch": mi["algorithmic_bytes"],
                        "batches": {"n": len(batch_gbs), "min_gbs": round(batch_gbs[0], 1),
                                    "median_gbs": round(batch_gbs[len(batch_gbs) // 2], 1),
                                    "max_gbs": round(batch_gbs[-1], 1),
                                    "median_frac": round(batch_gbs[len(batch_gbs) // 2] / HBM_PEAK_GBS, 4)}}}

    if not args.no_cpu:
        log("timing the reference CPU path")
        out["cpu_baseline"] = cpu_baseline(csr, x_host, y.cpu().numpy(), mi["algorithmic_bytes"])
    del csr, x, y
    torch.cuda.empty_cache()
    if not args.no_formats:
        out["formats"] = leg_formats(torch, tb, dev, args.steps)
    if not args.no_pagerank:
        out["pagerank"] = leg_pagerank(torch, tb, dev, cpu=not args.no_cpu)
        cpu_pr = out["pagerank"].pop("cpu_baseline", None)
        if out.get("cpu_baseline") and cpu_pr:
            out["cpu_baseline"]["pagerank"] = cpu_pr
        torch.cuda.empty_cache()
    if not args.no_batch:
        out["batch"] = leg_batch(torch, tb, dev)
        torch.cuda.empty_cache()
    if not args.no_adjoint:
        out["adjoint"] = leg_adjoint(torch, tb, dev)

    # the two targets in one place: SpMV at >= 70% of the HBM peak (CSR and
    # ELL), mixed-precision PageRank to 1e-10 at >= 1.6x the FP64 path
    tg = {"csr_pct_hbm_peak": out["config"]["pct_hbm_peak"]}
    if "formats" in out:
        tg["ell_pct_hbm_peak"] = round(100 * out["formats"]["ELL"]["gbs"] / HBM_PEAK_GBS, 2)
    if "pagerank" in out:
        var = out["pagerank"]["variants"]
        mixed = {k: v["speedup_vs_fp64"] for k, v in var.items() if k in ("f32", "bf16", "pattern_f32")}
        best = max(mixed, key=mixed.get)
        tg["pagerank_mixed_speedup_vs_fp64"] = mixed
        l1key = "l1_vs_oracle_pstar" if "l1_vs_oracle_pstar" in var[best] else "l1_vs_gpu_fp64_limit"
        tg["pagerank_mixed_best"] = {"variant": best, "speedup_vs_fp64": mixed[best], l1key: var[best][l1key]}
        # (the graph's columns hold one value each, so these read no stored values either)
        plain = {k: v for k, v in mixed.items() if k in ("f32", "bf16")}
        bs = max(plain, key=plain.get)
        tg["pagerank_f32_bf16_best"] = {"variant": bs, "speedup_vs_fp64": plain[bs], l1key: var[bs][l1key]}
    out["targets"] = tg

    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
