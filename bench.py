"""Benchmark of the TNF contig-graph path on one MI355X.

A step is one full pass of the pair stage over the 200,000-contig synthetic
metagenome (1,000 order-3 Markov genomes, log-normal lengths median 8 kb,
sigma 1.0, clipped to [1.5 kb, 500 kb], 0.5% N): the thresholded, per-row
capped edge list (cutoff 0.95, maxEdges 200) of all n(n-1)/2 pairs, from
HBM-resident FP32 TNF rows and FP64 log sizes.  The timed mode is the BF16
mode: an MFMA scan bounds every pair's distance from below in 28 projected
dimensions, the tiles it cannot rule out go through the BF16 Gram and the FP32
refinement; the exact FP32 mode and the FP16 mode run in the same process, and
their edge lists must be identical.

value = n(n-1)/2 / (seconds per step): effective pair evaluations per second.

Also reported: the learned proposal filter (MLP 136-256-256-32 trained on the
device for 20k steps on 10M pairs labelled by the exact path; k-means clusters
of the embeddings, each cluster paired with its 20 nearest (32 above 262,144
contigs), the BF16 TNF Gram and FP32 refinement within those cluster pairs)
with its edge recall against the exhaustive edge set; the launch shapes the
autotuner picks; the counting kernel's HBM throughput; CPU baselines on the host cores
(the reference's own openmp/TNF.cpp for counting when it is built next to the
oracle, the oracle's C restatement of gen_tnf_graph for pairs).
"""
from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys
import tempfile
import threading
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import mdet_amd as M  # noqa: E402
from mdet_amd import learned as L  # noqa: E402
from mdet_amd import workload as W  # noqa: E402

PEAK_BF16_TFLOPS = 2500.0  # MI355X dense BF16/FP16 MFMA
PEAK_HBM_GBS = 8000.0      # MI355X HBM3E
PEAK_FP32_UNPACKED_TFLOPS = 78.6  # the vector units without packed instructions, which this build leaves out
REFINE_FLOPS_PER_PAIR = 3 * 136  # FP32 squared distance: difference, product, sum per column
CUTOFF, MAX_EDGES = 0.95, 200

def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def run_mode(ctx, w, mode, steps, warmup):
    for _ in range(warmup):
        ctx.tnf_edges(w.tnf, w.logsize, w.n, CUTOFF, MAX_EDGES, mode, fetch=False)
    ctx.sync()
    stats = []
    t0 = time.perf_counter()
    for _ in range(steps):
        _, st = ctx.tnf_edges(w.tnf, w.logsize, w.n, CUTOFF, MAX_EDGES, mode, fetch=False)
        stats.append(st.as_dict())
    ctx.sync()
    dt = time.perf_counter() - t0
    return dt / steps, stats


def fetch_edges(ctx, w, mode):
    f, t, s, st = ctx.tnf_edges(w.tnf, w.logsize, w.n, CUTOFF, MAX_EDGES, mode)
    return f, t, s, st


def host_info():
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return {"cpu_model": model, "nproc": os.cpu_count(), "affinity": len(os.sched_getaffinity(0))}


def count_algorithmic_bytes(w):
    """Bytes the counting step must move: the 2-bit stream, the N-run list,
    the FP32 rows and the integer counts it writes."""
    return (w.n_bases + 3) // 4 + 16 * w.n_runs + 8 * (w.n + 1) + 2 * 136 * 4 * w.n


def time_count(ctx, w, reps=5):
    """Wall time of mdet_tnf_count on HBM-resident input (device-synchronised)."""
    out = []
    for _ in range(reps + 1):
        ctx.sync()
        t0 = time.perf_counter()
        ctx.tnf_count(w.packed, w.n_bases, w.runs, w.n_runs, w.base_off, w.n, w.counts, w.tnf)
        ctx.sync()
        out.append(time.perf_counter() - t0)
    return float(np.median(out[1:]))


def cpu_count_baseline(w, cfg_name, budget_contigs=30000):
    """openmp/TNF.cpp (built from the reference sources next to the oracle) on
    a FASTA of the first contigs of the same workload; its own timer around
    the TNF loop, which covers contigs of at least 2500 bases."""
    ref = os.path.join(ROOT, "oracle", "_ref", "tnf_ref")
    if not os.path.exists(ref):
        return None
    cfg = W.gen_config_of(cfg_name, seed=1)
    m = min(w.n, budget_contigs)
    threads = max(1, min(16, len(os.sched_getaffinity(0))))
    with tempfile.TemporaryDirectory() as td:
        fa = os.path.join(td, "sample.fa")
        with open(fa, "wb") as f:
            for c in range(m):
                f.write(b">c%d\n" % c)
                f.write(M.gen_ascii(cfg, c, int(w.lengths[c])))
                f.write(b"\n")
        r = subprocess.run([ref, str(threads), fa], cwd=td, capture_output=True, text=True, timeout=600)
    secs = None
    for line in r.stdout.splitlines():
        if line.startswith("Crear matriz TNF"):
            secs = float(line.split()[-1].rstrip("s"))
    if r.returncode != 0 or secs is None:
        return None
    lens = w.lengths[:m]
    bases = int(lens[lens >= 2500].sum())
    return {"value": bases / secs, "unit": "bases/s", "cores": threads, "kind": "reference",
            "build": "g++ -O3 -march=x86-64-v3 -fopenmp openmp/TNF.cpp -lz (oracle/Makefile target ref)",
            "sample": f"first {m} contigs of the workload as FASTA ({bases} bases in contigs >= 2500, the ones "
                      f"openmp/TNF.cpp counts), its own timer around the TNF loop: {secs:.3f} s"}


def run_learned(ctx, w, fb, tb, train_steps, steps, n_probe, quantile=0.9999, autotune=True, use_radius=False,
                knn_study=False):
    """Train the filter on pairs the exact path labels, then time the learned
    edge list (cluster index over the embeddings, n_probe nearest clusters;
    within the probed cluster pairs the BF16 TNF Gram decides, or with
    use_radius the embedding radius) and measure its recall against the
    exhaustive edge set."""
    n = w.n
    # training in the library (mdet_mlp_fit): standardisation, labels from
    # one exact BF16-refine call, the 1:4 training set and the Adam steps
    mlp = M.Mlp(ctx, seed=7)
    fit, curve = mlp.fit(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, n_pairs=10_000_000, steps=train_steps, batch=512,
                         lr=2e-3, margin=4.0, seed=1, radius_quantile=quantile if use_radius else 0.0,
                         loss_every=max(1, train_steps // 10))
    rec = ctx.last_pairs()  # the labelling call's exactly decided pairs
    pos = rec[(rec["flags"] & 2) != 0]
    r2 = fit["radius2"] if use_radius else 0.0
    kw = dict(mlp=mlp, radius2=r2, n_probe=n_probe)
    tune = ctx.autotune(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, reps=2, **kw) if autotune \
        else ctx.tune_get(M.LEARNED)
    for _ in range(2):
        ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw)
    ctx.sync()
    stats = []
    t0 = time.perf_counter()
    for _ in range(steps):
        _, st = ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw)
        stats.append(st.as_dict())
    ctx.sync()
    sec = (time.perf_counter() - t0) / steps
    f, t, s, st = ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, **kw)
    exact = fb.astype(np.uint64) * n + tb.astype(np.uint64)
    got = f.astype(np.uint64) * n + t.astype(np.uint64)
    hit = np.isin(exact, got)
    # the same network without the full-row fallback (faster; a missed partner of a full row lets
    # the next proposed one in)
    ctx.set_learned_fallback(False)
    ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw)
    ctx.sync()
    t0 = time.perf_counter()
    for _ in range(3):
        ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw)
    ctx.sync()
    nofb_sec = (time.perf_counter() - t0) / 3
    fn, tn, _, _ = ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, **kw)
    ctx.set_learned_fallback(True)
    gotn = fn.astype(np.uint64) * n + tn.astype(np.uint64)
    no_fallback = {"ms_per_step": nofb_sec * 1e3, "speedup_vs_bf16_refine": None,
                   "edge_recall": float(np.isin(exact, gotn).mean()) if len(exact) else 1.0,
                   "edges_not_in_exhaustive_set": int((~np.isin(gotn, exact)).sum())}
    # the exact cover: cluster pairs from the TNF-space triangle bound (clusters of a fixed sign
    # projection of the TNF rows, no network, no probes, no full-row step); its edge list must be
    # the exhaustive one
    ctx.set_learned_exact_cover(True)
    kw_cov = dict(mlp=None, radius2=0.0, n_probe=1)
    try:
        for _ in range(2):
            ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw_cov)
        ctx.sync()
        t0 = time.perf_counter()
        for _ in range(steps):
            ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw_cov)
        ctx.sync()
        cov_sec = (time.perf_counter() - t0) / steps
        fc, tc, _, stc = ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, **kw_cov)
    finally:
        ctx.set_learned_exact_cover(False)
    exact_cover = {"ms_per_step": cov_sec * 1e3, "speedup_vs_bf16_refine": None,
                   "pairs_per_s": n * (n - 1) // 2 / cov_sec, "candidate_pairs": int(stc.pairs_evaluated),
                   "candidate_fraction": stc.pairs_evaluated / max(1, n * (n - 1) // 2),
                   "survivors_exact_evaluated": int(stc.survivors),
                   "edge_list_identical_to_exhaustive": bool(np.array_equal(fc, fb) and np.array_equal(tc, tb)),
                   "full_rows_completed": int(stc.fallback_rows),
                   "clusters": "n/128 k-means clusters of a fixed sign projection of the TNF rows"}
    # the per-row top-k form of the filter (k nearest embedding neighbours per column tile), measured
    # by brute force for comparison with the cluster index
    knn_points = [(128, 0), (256, 0), (512, 0), (256, n // 4), (64, n // 16)] if knn_study else []
    knn = {"trained": [L.knn_candidate_recall(L.embeddings(ctx, mlp, w.tnf, n), exact, k, t_)
                       for k, t_ in knn_points]} if knn_points else {}
    mlp.close()
    # the same filter with an untrained network (what the training buys)
    raw = M.Mlp(ctx, seed=7)
    raw.norm_from_rows(w.tnf, n)
    kw_raw = dict(kw, mlp=raw)
    if use_radius:
        kw_raw["radius2"] = L.calibrate_radius2(L.embeddings(ctx, raw, w.tnf, n), pos["i"], pos["j"],
                                                quantile=quantile)
    ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw_raw)
    ctx.sync()
    t0 = time.perf_counter()
    for _ in range(3):
        ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw_raw)
    ctx.sync()
    raw_sec = (time.perf_counter() - t0) / 3
    fr, tr, _, str_ = ctx.tnf_edges(w.tnf, w.logsize, n, CUTOFF, MAX_EDGES, M.LEARNED, **kw_raw)
    raw_hit = np.isin(exact, fr.astype(np.uint64) * n + tr.astype(np.uint64))
    if knn_points:
        raw_emb = L.embeddings(ctx, raw, w.tnf, n)
        knn["untrained"] = [L.knn_candidate_recall(raw_emb, exact, k, t_) for k, t_ in knn_points]
    raw.close()
    untrained = {"ms_per_step": raw_sec * 1e3, "candidate_pairs": str_.pairs_evaluated,
                 "full_rows_completed_exactly": int(str_.fallback_rows), "fallback_pairs": int(str_.fallback_pairs),
                 "edges_not_in_exhaustive_set": int((~np.isin(fr.astype(np.uint64) * n + tr.astype(np.uint64),
                                                              exact)).sum()),
                 "survivors_exact_evaluated": str_.survivors,
                 "edge_recall": float(raw_hit.mean()) if len(exact) else 1.0}
    return {"pairs_per_s": n * (n - 1) // 2 / sec, "ms_per_step": sec * 1e3,
            "stage_ms": {k: float(np.mean([x[k] for x in stats]))
                         for k in ("ms_prefilter", "ms_refine", "ms_select", "ms_total")},
            "candidate_pairs": stats[-1]["pairs_evaluated"], "n_probe": n_probe,
            "survivors_exact_evaluated": stats[-1]["survivors"], "edges": int(len(f)),
            "edge_recall": float(hit.mean()) if len(exact) else 1.0,
            "edges_not_in_exhaustive_set": int((~np.isin(got, exact)).sum()),
            "rows_capped": int(st.rows_capped),
            "full_rows_completed_exactly": int(st.fallback_rows),
            "fallback_pairs": int(st.fallback_pairs),
            "within_cluster_pairs": "embedding radius" if use_radius else "BF16 TNF Gram prefilter",
            "untrained_network_same_probes": untrained,
            "without_full_row_fallback": no_fallback,
            "exact_cover": exact_cover,
            **({"per_row_topk_form": knn} if knn_points else {}),
            "radius2": r2, "radius_quantile": quantile if use_radius else None, "tune": tune,
            "training": {"api": "mdet_mlp_fit", "pairs": int(fit["pairs"]), "positives": int(fit["positives"]),
                         "labelled": int(fit["labelled"]), "steps": train_steps, "batch": 512,
                         "seconds": fit["ms_train"] / 1e3, "ms_per_step": fit["ms_train"] / max(1, train_steps),
                         "set_build_s": fit["ms_label"] / 1e3, "loss_curve": curve}}


def copy_probe(mib):
    """A plain device copy of known size (elementwise y = 2x, mib MiB each way),
    for scaling the FETCH_SIZE / WRITE_SIZE counters."""
    import torch
    x = torch.ones(mib * (1 << 20) // 4, dtype=torch.float32, device="cuda")
    y = torch.empty_like(x)
    for _ in range(3):
        torch.mul(x, 2.0, out=y)
    torch.cuda.synchronize()
    print(json.dumps({"copy_probe_bytes_each_way": mib << 20, "kernel": "elementwise mul"}))


def gemm_probe():
    """The dense BF16 MFMA rate this GPU sustains in a library GEMM
    (torch.matmul on hipBLASLt, M = N = K = 8192, and the Gram shape of the
    prefilter, K = 144, whose M x M output makes it write-bound), for reading
    the prefilter's fraction of the published peak."""
    import torch
    out = {}
    for m, k in ((8192, 8192), (16384, 144)):
        a = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
        b = torch.randn(k, m, device="cuda", dtype=torch.bfloat16)
        for _ in range(5):
            c = torch.matmul(a, b)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        reps = 50
        e0.record()
        for _ in range(reps):
            c = torch.matmul(a, b)
        e1.record()
        torch.cuda.synchronize()
        ms = e0.elapsed_time(e1) / reps
        tflops = 2.0 * m * m * k / (ms * 1e-3) / 1e12
        out[f"m{m}_k{k}"] = {"ms": ms, "TFLOP/s": tflops, "frac_of_2500": tflops / PEAK_BF16_TFLOPS,
                             "output_GB/s": m * m * c.element_size() / (ms * 1e-3) / 1e9}
        del a, b, c
    print(json.dumps({"gemm_probe": out, "dtype": "bf16", "library": "torch.matmul (hipBLASLt)"}))


def build_pair_baseline(tmpdir):
    """The OpenMP pair baseline (oracle/pair_baseline.c over the oracle's
    restatement of gen_tnf_graph), compiled on this machine with -O3
    -march=native -fopenmp; returns (ctypes library, flags)."""
    import ctypes as C
    subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "oracle"), "base", f"BASEDIR={tmpdir}"], check=True)
    flags = subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "oracle"), "print-pairbase-flags"],
                           capture_output=True, text=True, check=True).stdout.strip()
    lib = C.CDLL(os.path.join(tmpdir, "libpairbase.so"))
    P = np.ctypeslib.ndpointer
    lib.pairbase_rows.argtypes = [P(np.float32, flags="C"), P(np.float64, flags="C"), C.c_size_t, C.c_double,
                                  C.c_size_t, C.c_size_t, C.c_size_t, P(np.uint32, flags="C"),
                                  P(np.uint64, flags="C"), C.c_int]
    lib.pairbase_rows.restype = C.c_int
    return lib, flags


def cpu_baseline(tnf, ls, fb, tb, budget_s=12.0):
    """The oracle's per-row scan of gen_tnf_graph (every column of each row,
    the FP64 model, the per-row heap) built -O3 -march=native -fopenmp and run
    with one OpenMP thread per host core on a leading row sample; its per-row
    edge counts and partner-id sums are compared with the GPU edge list."""
    n = tnf.shape[0]
    threads = max(1, min(16, len(os.sched_getaffinity(0))))
    tnf = np.ascontiguousarray(tnf, np.float32)
    ls = np.ascontiguousarray(ls, np.float64)
    with tempfile.TemporaryDirectory() as td:
        lib, flags = build_pair_baseline(td)
        cnt = np.zeros(n, np.uint32)
        sj = np.zeros(n, np.uint64)
        # calibrate on a few rows, then size the timed sample to the budget
        t0 = time.perf_counter()
        lib.pairbase_rows(tnf, ls, n, CUTOFF, MAX_EDGES, 0, 4 * threads, cnt, sj, threads)
        per_row = (time.perf_counter() - t0) / (4 * threads)
        rows = int(min(n, max(8 * threads, budget_s / per_row)))
        t0 = time.perf_counter()
        used = lib.pairbase_rows(tnf, ls, n, CUTOFF, MAX_EDGES, 0, rows, cnt, sj, threads)
        dt = time.perf_counter() - t0
    pairs = rows * (n - 1)
    m = fb < rows
    g_cnt = np.bincount(fb[m], minlength=rows)[:rows]
    g_sj = np.bincount(fb[m], weights=tb[m].astype(np.float64), minlength=rows)[:rows]
    same = bool(np.array_equal(g_cnt, cnt[:rows]) and np.array_equal(g_sj.astype(np.uint64), sj[:rows]))
    return {"value": pairs / dt, "unit": "pairs/s", "cores": int(used), "kind": "port",
            "build": f"gcc {flags} (oracle/pair_baseline.c, built on this host)",
            "sample": f"rows 0..{rows - 1} of {n} against all {n} columns ({pairs:.3g} ordered pairs, "
                      f"{dt:.1f} s): gen_tnf_graph's per-row scan with the FP64 model and heap"}, same, rows


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--workload", default="c3_200k", choices=sorted(W.CONFIGS))
    ap.add_argument("--n", type=int, default=None, help="override the contig count")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--modes", default="exact_f32,f16_refine")
    ap.add_argument("--train-steps", type=int, default=20000)
    ap.add_argument("--no-learned", action="store_true")
    ap.add_argument("--learned-radius", action="store_true",
                    help="learned filter: embedding radius test within the probed cluster pairs "
                         "(default: the BF16 TNF Gram decides there)")
    ap.add_argument("--knn-study", action="store_true",
                    help="also measure the per-row top-k form of the learned filter (k nearest embedding "
                         "neighbours per column tile, brute force) for the trained and untrained network")
    ap.add_argument("--no-autotune", action="store_true",
                    help="time the BF16 and learned paths at the default launch shapes")
    ap.add_argument("--n-probe", type=int, default=0,
                    help="clusters probed per cluster by the learned filter (0: 20 up to 262,144 contigs, else 32)")
    ap.add_argument("--gemm-probe", action="store_true",
                    help="time a dense BF16 library GEMM (the achievable MFMA rate) and exit")
    ap.add_argument("--copy-probe-mib", type=int, default=0,
                    help="only run a plain copy of this size (counter calibration) and exit")
    ap.add_argument("--count-only", action="store_true",
                    help="only time the counting step on the workload (profiling runs) and exit")
    ap.add_argument("--cover-only", action="store_true",
                    help="only time the learned mode's exact cover on the workload against one BF16-refine "
                         "call (profiling runs) and exit")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU; --gpus must be 1"}))
        sys.exit(2)
    if args.gemm_probe:
        gemm_probe()
        return
    if args.copy_probe_mib:
        copy_probe(args.copy_probe_mib)
        return

    if args.knn_study:
        # torch's HIP runtime has to claim the device before the library's context does
        import torch
        torch.cuda.init()
    ctx = M.Ctx(0)
    log(f"generating {args.workload}")
    w = W.make(ctx, args.workload, n=args.n, seed=1, keep_stream=True)
    log(f"{w.n} contigs, {w.n_bases} bases, generated in {w.gen_s:.1f} s, counted in {w.count_ms:.1f} ms")
    P = w.n * (w.n - 1) // 2
    count_s = time_count(ctx, w)
    count_bytes = count_algorithmic_bytes(w)
    count = {"bases_per_s": w.n_bases / count_s, "ms": count_s * 1e3, "algorithmic_bytes": count_bytes,
             "achieved_GBs": count_bytes / count_s / 1e9, "peak_GBs": PEAK_HBM_GBS,
             "frac": count_bytes / count_s / 1e9 / PEAK_HBM_GBS,
             "note": "wall time of mdet_tnf_count (counting + normalisation kernels, host checks) on resident input"}
    if args.count_only:
        print(json.dumps({"workload": args.workload, "n_contigs": w.n, "n_bases": w.n_bases, "n_runs": w.n_runs,
                          "count": count}))
        ctx.close()
        return
    for a in (w.packed, w.runs, w.base_off):
        a.free()
    if args.cover_only:
        fb, tb, _, stb = ctx.tnf_edges(w.tnf, w.logsize, w.n, CUTOFF, MAX_EDGES, M.BF16_REFINE)
        ctx.set_learned_exact_cover(True)
        kw = dict(mlp=None, radius2=0.0, n_probe=1)
        for _ in range(args.warmup):
            ctx.tnf_edges(w.tnf, w.logsize, w.n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw)
        ctx.sync()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            ctx.tnf_edges(w.tnf, w.logsize, w.n, CUTOFF, MAX_EDGES, M.LEARNED, fetch=False, **kw)
        ctx.sync()
        sec = (time.perf_counter() - t0) / args.steps
        fc, tc, _, stc = ctx.tnf_edges(w.tnf, w.logsize, w.n, CUTOFF, MAX_EDGES, M.LEARNED, **kw)
        print(json.dumps({"workload": args.workload, "n_contigs": w.n, "exact_cover_ms": sec * 1e3,
                          "bf16_refine_ms_one_call": stb.ms_total, "candidate_pairs": int(stc.pairs_evaluated),
                          "edge_list_identical_to_exhaustive": bool(np.array_equal(fc, fb) and np.array_equal(tc, tb))}))
        ctx.close()
        return

    # headline: the BF16 mode, at the launch shape the autotuner picks for this input
    if args.no_autotune:
        tune = ctx.tune_get(M.BF16_REFINE)
    else:
        log("autotuning bf16_refine")
        tune = ctx.autotune(w.tnf, w.logsize, w.n, CUTOFF, MAX_EDGES, M.BF16_REFINE, reps=2)
        log(f"  {tune}")
    log("timing bf16_refine")
    sec, stats = run_mode(ctx, w, M.BF16_REFINE, args.steps, args.warmup)
    pf_ms = float(np.mean([s["ms_prefilter"] for s in stats]))
    modes = {"bf16_refine": {"pairs_per_s": P / sec, "ms_per_step": sec * 1e3,
                             "stage_ms": {k: float(np.mean([s[k] for s in stats]))
                                          for k in ("ms_prefilter", "ms_refine", "ms_select", "ms_total")},
                             "survivors": stats[-1]["survivors"], "candidates": stats[-1]["candidates"],
                             "adjudicated_fp64": stats[-1]["adjudicated"], "tune": tune}}
    fb, tb, sb, stb = fetch_edges(ctx, w, M.BF16_REFINE)
    modes["bf16_refine"]["edges"] = int(len(fb))
    modes["bf16_refine"]["rows_capped"] = int(stb.rows_capped)
    modes["bf16_refine"]["rows_block_select"] = int(stb.rows_block)
    modes["bf16_refine"]["rows_global_select"] = int(stb.rows_global)
    # every emitted FP32 similarity against its FP64 value (the reference's double sTNF)
    s64 = ctx.tnf_similarity64(w.tnf, w.logsize, w.n, fb, tb)
    modes["bf16_refine"]["max_abs_s_err_vs_fp64"] = float(np.max(np.abs(sb.astype(np.float64) - s64))) \
        if len(fb) else 0.0
    del s64

    identical = {}
    for name in [m for m in args.modes.split(",") if m]:
        mode = M.PRECISIONS[name]
        steps = max(1, args.steps // 3)
        log(f"timing {name} ({steps} steps)")
        sec_m, st_m = run_mode(ctx, w, mode, steps, 1)
        f, t, s, _ = fetch_edges(ctx, w, mode)
        same = bool(np.array_equal(f, fb) and np.array_equal(t, tb))
        identical[name] = same
        modes[name] = {"pairs_per_s": P / sec_m, "ms_per_step": sec_m * 1e3,
                       "stage_ms": {k: float(np.mean([x[k] for x in st_m]))
                                    for k in ("ms_prefilter", "ms_refine", "ms_select", "ms_total")},
                       "edges": int(len(f)), "edge_set_identical_to_bf16": same,
                       "max_abs_s_diff_vs_bf16": float(np.max(np.abs(s - sb))) if same and len(s) else None}
    if "exact_f32" in modes:
        modes["bf16_refine"]["speedup_vs_exact_f32"] = modes["bf16_refine"]["pairs_per_s"] / modes["exact_f32"]["pairs_per_s"]
    if not args.no_learned:
        log(f"learned filter: {args.train_steps} training steps")
        n_probe = args.n_probe or (20 if w.n <= 262144 else 32)
        lm = run_learned(ctx, w, fb, tb, args.train_steps, args.steps, n_probe, autotune=not args.no_autotune,
                         use_radius=args.learned_radius, knn_study=args.knn_study)
        lm["speedup_vs_bf16_refine"] = lm["pairs_per_s"] / modes["bf16_refine"]["pairs_per_s"]
        nf = lm["without_full_row_fallback"]
        nf["speedup_vs_bf16_refine"] = modes["bf16_refine"]["ms_per_step"] / nf["ms_per_step"]
        ec = lm["exact_cover"]
        ec["speedup_vs_bf16_refine"] = modes["bf16_refine"]["ms_per_step"] / ec["ms_per_step"]
        modes["learned"] = lm

    # the second pass takes the largest share of a step: the Gram of the listed
    # tiles, and the FP32 distance and model of every survivor (k_tile_refine,
    # bound by the vector units' issue slots); only the distances are counted
    ref_ms = modes["bf16_refine"]["stage_ms"]["ms_refine"]
    flops = REFINE_FLOPS_PER_PAIR * modes["bf16_refine"]["survivors"]
    achieved = flops / (ref_ms * 1e-3) / 1e12
    roofline = {"bound": "valu", "kernel": "k_tile_refine (with k_tile_gram and k_adjudicate)", "achieved": achieved,
                "peak": PEAK_FP32_UNPACKED_TFLOPS, "unit": "TFLOP/s", "frac": achieved / PEAK_FP32_UNPACKED_TFLOPS,
                "flops_per_step": flops, "avg_stage_ms": ref_ms, "scan_ms": pf_ms,
                "timing": "HIP events recorded on the context stream around the stage, mean of the timed steps"}

    cpu = None
    cpu_count = None
    parity = {}
    if not args.no_cpu:
        log("cpu baseline (oracle pair scan, -O3 -march=native -fopenmp, row sample)")
        tnf, ls = w.tnf.numpy(), w.logsize.numpy()
        cpu, same, rows = cpu_baseline(tnf, ls, fb, tb)
        cpu.update(host_info())
        log("cpu counting baseline (openmp/TNF.cpp)")
        cpu_count = cpu_count_baseline(w, args.workload)
        if cpu_count:
            cpu_count.update(host_info())
        parity = {"oracle_rows_checked": rows, "edges_in_rows_equal_oracle": same,
                  "compared": "per-row edge count and partner-id sum of the BF16 list against the CPU scan"}

    line = {
        "metric": "TNF pair evals/s: exact vs BF16-refine vs learned filter at >=99.9% edge recall",
        "value": P / sec,
        "unit": "pairs/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": sec * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic",
        "config": {"workload": f"{args.workload}: {w.n} contigs, {W.CONFIGS[args.workload]['n_genomes']} genomes, "
                               f"{w.n_bases} bases; cutoff {CUTOFF}, maxEdges {MAX_EDGES}; step = full edge list "
                               f"of {P} pairs (bf16_refine)",
                   "n_contigs": w.n, "pairs": P, "cutoff": CUTOFF, "max_edges": MAX_EDGES,
                   "count_ms": count["ms"], "count_bases_per_s": count["bases_per_s"]},
        "modes": modes,
        "count": count,
        "edge_sets_identical": identical,
        "parity": parity,
        "roofline": roofline,
        "cpu_baseline": cpu,
        "cpu_baseline_count": cpu_count,
    }
    print(json.dumps(line))
    ctx.close()


if __name__ == "__main__":
    main()
