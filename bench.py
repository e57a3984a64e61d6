"""All-vs-all cRMSD throughput on one MI355X.

Workload (the headline configuration): one ensemble of 10,000 conformations x
300 CA atoms, 5 % near-identical (sigma 0.01 A), the rest sigma ~ U(0.5, 4) A,
generated deterministically on the host and copied to HBM before timing.  A
step is one all-vs-all pass: per-conformation preparation, the BF16x3 Gram
MFMA kernel with the fused FP64 QCP epilogue, and FP64 re-evaluation of
flagged pairs, writing the 49,995,000-value packed f32 triangle to HBM.

Also measured in the same run: the plain per-pair GPU kernel (FP32) on the
same input, the error of both against the FP64 oracle on a row sample, and the
oracle itself on the host cores (cpu_baseline, a bounded row sample).  More
legs report the neighbouring workloads beside the headline line: "batch" (512
ensembles of uneven n and L as one graph launch, autotuned tiles), "serving"
(query-vs-library top-100 over device-resident libraries, Poisson arrivals at
a fixed rate, p50/p99 latency and pairs/s) and "next" (clustering, row
reductions, superposition output, ingestion and the TSV writer).

Prints one JSON line.
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

METRIC = "superpositions/s all-vs-all N=10k L=300 vs plain GPU; p50/p99 ms at fixed QPS"
PEAK_BF16_TFLOPS = 2500.0  # MI355X dense BF16 MFMA
PEAK_FP32_VALU_TFLOPS = 157.3
PEAK_FP64_VALU_TFLOPS = 78.6


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


def pmc_figure(n: int, L: int, key: str) -> float | None:
    """A figure of the committed rocprofv3 --pmc summary of the 10,000 x 300 Gram
    launch (a `key = value` line), or None for other shapes or when absent."""
    path = os.path.join(ROOT, "profiles", "gram_bf16x3_10k_300_pmc.txt")
    if (n, L) != (10000, 300) or not os.path.exists(path):
        return None
    with open(path) as f:
        for line in f:
            if line.startswith(key + " "):
                return float(line.split("=")[1].split()[0])
    return None


def traffic_bytes(n: int, L: int) -> int | None:
    """HBM bytes per Gram launch: FETCH_SIZE and WRITE_SIZE, each scaled by the factor
    the same counter reads for a device copy of known size."""
    v = pmc_figure(n, L, "traffic_bytes_per_launch")
    return None if v is None else int(v)


def measured_peaks() -> dict:
    """Dense BF16 MFMA and FP64 FMA rates this GPU sustains in a probe kernel
    (reference points only; every frac uses the published peak)."""
    import ctypes

    from bioshell_amd import _native

    f = _native.diag_lib().bsi_peak_probe
    f.argtypes = [ctypes.c_int, ctypes.POINTER(ctypes.c_double)]
    f.restype = ctypes.c_int
    out = {}
    for which, key in ((0, "bf16_mfma_tflops"), (1, "fp64_fma_tflops")):
        v = ctypes.c_double(0.0)
        rc = f(which, ctypes.byref(v))
        out[key] = round(v.value, 1) if rc == 0 else None
    out["probe"] = ("back-to-back v_mfma_f32_32x32x16_bf16 on 8 accumulators per wave, and 16 FP64 FMA "
                    "chains per lane, all CUs, best of 3 runs of ~1 ms")
    return out


def batch_leg(args, B, torch, log) -> dict:
    """512 independent ensembles, n ~ U(20, 500), L ~ U(30, 800), sigma ~ U(0.5, 3):
    autotuned tiles, the whole batch as one graph launch, inputs resident in HBM."""
    from oracle import oracle as O

    rng = np.random.default_rng(3)
    E = args.batch_ensembles
    ns = rng.integers(20, 501, E)
    Ls = rng.integers(30, 801, E)
    log(f"batch: generating {E} ensembles ({int((ns * Ls).sum() * 24) >> 20} MiB)")
    xs = [B.generate_ensemble(7000 + e, int(ns[e]), int(Ls[e]), sigma=(0.5, 3.0)) for e in range(E)]
    pairs = int(sum(n * (n - 1) // 2 for n in ns))
    dev = torch.device("cuda:0")
    d_in = [torch.from_numpy(x).to(dev) for x in xs]
    d_out = [torch.empty(int(n) * (int(n) - 1) // 2, dtype=torch.float32, device=dev) for n in ns]
    torch.cuda.synchronize()
    ctx = B.Context(0)
    t0 = time.perf_counter()
    ctx.autotune(B.Method.BF16X3_GRAM, None)
    tune_s = time.perf_counter() - t0
    ptr_in = [t.data_ptr() for t in d_in]
    ptr_out = [t.data_ptr() for t in d_out]

    def step(method):
        B.crmsd_batch_device(ptr_in, ns, Ls, ptr_out, method, ctx=ctx)

    t0 = time.perf_counter()
    step(B.Method.BF16X3_GRAM)  # builds the graph
    torch.cuda.synchronize()
    first_ms = (time.perf_counter() - t0) * 1e3
    for _ in range(args.warmup):
        step(B.Method.BF16X3_GRAM)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step(B.Method.BF16X3_GRAM)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / args.steps
    dev_ms = float(np.median([h["total_ms"] for h in ctx.history(args.steps)]))
    flagged = int(ctx.last_stats()["flagged_pairs"])
    log(f"batch bf16x3: {dt * 1e3:.3f} ms/step (device {dev_ms:.3f} ms), {pairs} pairs")
    got = [t.cpu().numpy() for t in d_out]
    # error against the oracle on the 8 ensembles with the fewest pairs x atoms
    order = np.argsort(ns * ns * Ls)[:8]
    err = max(float(np.abs(got[e].astype(np.float64) - O.all_vs_all(xs[e])).max()) for e in order)
    # plain per-pair kernel over the same batch (one launch per ensemble)
    step(B.Method.FP32_PLAIN)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(2):
        step(B.Method.FP32_PLAIN)
    torch.cuda.synchronize()
    plain_dt = (time.perf_counter() - t0) / 2
    # host buffers in and out (PCIe and staging included)
    t0 = time.perf_counter()
    B.crmsd_batch(xs, B.Method.BF16X3_GRAM, ctx=ctx)
    host_dt = time.perf_counter() - t0
    ctx.close()
    return {
        "workload": f"{E} ensembles, n ~ U(20,500), L ~ U(30,800), sigma U(0.5,3) A; "
                    "BF16X3_GRAM, autotuned tiles, one graph launch per batch",
        "pairs": pairs,
        "value": round(pairs / dt, 1),
        "unit": "superpositions/s",
        "ms_per_step": round(dt * 1e3, 3),
        "device_ms_per_step": round(dev_ms, 3),
        "first_call_ms_incl_graph_build": round(first_ms, 2),
        "autotune_s": round(tune_s, 2),
        "flagged_pairs": flagged,
        "max_abs_err_vs_fp64_8_ensembles": err,
        "plain_fp32_ms_per_step": round(plain_dt * 1e3, 3),
        "speedup_vs_plain": round(plain_dt / dt, 2),
        "host_io_ms_per_call": round(host_dt * 1e3, 1),
    }


def serving_leg(args, B, log) -> dict:
    """Device-resident libraries of 25,000 conformations in each of L = 64, 128,
    256, 512; Poisson arrivals at a fixed rate; each request 1-64 queries of one
    bucket, top-100 lowest cRMSD."""
    buckets = (64, 128, 256, 512)
    n_lib = args.serve_library
    ctx = B.Context(0)
    libs, pools = [], []
    for b, L in enumerate(buckets):
        x = B.generate_ensemble(8000 + b, n_lib + 256, L, sigma=(0.5, 3.0))
        libs.append(B.Library(x[:n_lib], ctx=ctx))
        pools.append(np.ascontiguousarray(x[n_lib:]))
    log(f"serving: libraries ready ({len(buckets)} x {n_lib})")
    srv = B.Server(libs, max_inflight=4)
    rng = np.random.default_rng(11)
    R = args.serve_requests
    gaps = rng.exponential(1.0 / args.serve_qps, R)
    reqs = []
    for _ in range(R):
        b = int(rng.integers(0, len(buckets)))
        nq = int(rng.integers(1, 65))
        s0 = int(rng.integers(0, 256 - nq + 1))
        reqs.append((b, pools[b][s0:s0 + nq]))
    # warm every slot and kernel: four concurrent requests per bucket
    for b in range(len(buckets)):
        warm = [srv.submit(b, pools[b][:64], 100) for _ in range(4)]
        for t in warm:
            t.wait()
    tickets = []
    t_start = time.perf_counter()
    due = t_start
    for (b, q), g in zip(reqs, gaps):
        due += g
        while True:
            now = time.perf_counter()
            if now >= due:
                break
            if due - now > 0.002:
                time.sleep(due - now - 0.001)
        tickets.append(srv.submit(b, q, 100))
    for t in tickets:
        t.wait()
    wall = time.perf_counter() - t_start
    lat = np.array([t.latency_ms() for t in tickets])
    pairs = sum(q.shape[0] for _, q in reqs) * n_lib
    # capacity: the same requests submitted at once (queueing dominates latency)
    t0 = time.perf_counter()
    burst = [srv.submit(b, q, 100) for b, q in reqs]
    for t in burst:
        t.wait()
    sat = time.perf_counter() - t0
    srv.close()
    for l in libs:
        l.close()
    ctx.close()
    log(f"serving: p50 {np.percentile(lat, 50):.3f} ms, p99 {np.percentile(lat, 99):.3f} ms")
    return {
        "workload": f"libraries of {n_lib} conformations at L = 64/128/256/512 (resident in HBM); "
                    f"Poisson arrivals at {args.serve_qps} requests/s; 1-64 queries of one bucket "
                    "per request; top-100",
        "requests": R,
        "qps_offered": args.serve_qps,
        "qps_achieved": round(R / wall, 1),
        "p50_ms": round(float(np.percentile(lat, 50)), 3),
        "p99_ms": round(float(np.percentile(lat, 99)), 3),
        "mean_ms": round(float(lat.mean()), 3),
        "pairs_per_s": round(pairs / wall, 1),
        "latency": "submit to host-visible top-100 (bs_server_latency_ms)",
        "capacity_requests_per_s": round(R / sat, 1),
        "capacity_pairs_per_s": round(pairs / sat, 1),
    }


def synthetic_cif(n_models: int) -> bytes:
    """A multi-model mmCIF text: the 255 atoms of the first 2jqb model (the
    reference's multi-model fixture) repeated as n_models models, each with
    its coordinates displaced."""
    from oracle import ingest_oracle as I

    raw = I.read_text(os.path.join(ROOT, "tests", "golden", "structures", "2jqb.cif.gz")).decode()
    head, rest = raw.split("_atom_site.pdbx_PDB_model_num", 1)
    body, tail = rest.split("\n#", 1)
    first = [l.split() for l in body.split("\n") if l.strip() and l.split()[-1] == "1"]
    rng = np.random.default_rng(1)
    out = [head, "_atom_site.pdbx_PDB_model_num\n"]
    for m in range(n_models):
        d = rng.normal(size=(len(first), 3)) * 0.5
        for t, dd in zip(first, d):
            t = list(t)
            t[-1] = str(m + 1)
            for c in range(3):
                t[10 + c] = f"{float(t[10 + c]) + dd[c]:.3f}"
            out.append(" ".join(t) + "\n")
    out.append("#" + tail)
    return "".join(out).encode()


def stream_ms(torch, ctx, fn, reps: int) -> tuple[float, float]:
    """(device ms, host ms) per call of fn over reps calls, after one untimed
    call.  Device time is HIP events recorded on the context's own stream, the
    stream the library launches on (torch's current stream would see none of it);
    host time also holds the launch overhead of each call."""
    s = torch.cuda.ExternalStream(ctx.stream)
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    fn()
    ctx.synchronize()
    t0 = time.perf_counter()
    a.record(s)
    for _ in range(reps):
        fn()
    b.record(s)
    b.synchronize()
    host = (time.perf_counter() - t0) * 1e3 / reps
    return a.elapsed_time(b) / reps, host


def next_rows_leg(args, B, torch, log, ctx, d_xyz, d_out, x) -> dict:
    """The path's neighbours, each on its own workload: clustering and row
    reductions over the headline triangle already in HBM, ensemble superposition
    of the headline ensemble, ensemble ingestion from mmCIF text, and the clust
    TSV writer.  CPU figures are the oracle (or single-threaded native code where
    the oracle has no counterpart) on a bounded sample, as stated per entry."""
    from bioshell_amd import clustering as C
    from oracle import ingest_oracle as I
    from oracle import oracle as O

    n, L = x.shape[:2]
    out = {}
    dev = d_out.device
    # ---- row minima / maxima (outliers, medoid) and clustering, triangle in HBM
    d_lo = torch.empty(n, dtype=torch.float32, device=dev)
    d_hi = torch.empty(n, dtype=torch.float32, device=dev)
    import ctypes

    from bioshell_amd import _native

    vp = ctypes.c_void_p
    reps = 20

    def row_stats():
        B.check(_native.lib().bs_rmsd_row_stats_device(ctx.handle, vp(d_out.data_ptr()), n, vp(d_lo.data_ptr()),
                                                        vp(d_hi.data_ptr())))

    rs_ms, rs_host_ms = stream_ms(torch, ctx, row_stats, reps)
    tri_bytes = n * (n - 1) // 2 * 4
    # the same statistics taken in the Gram epilogue, against the all-vs-all alone
    d_lo2 = torch.empty(n, dtype=torch.float32, device=dev)
    d_hi2 = torch.empty(n, dtype=torch.float32, device=dev)
    gram = int(B.Method.BF16X3_GRAM)

    def avsa():
        B.check(_native.lib().bs_crmsd_all_vs_all_device(ctx.handle, vp(d_xyz.data_ptr()), n, L, gram,
                                                          vp(d_out.data_ptr()), 0))

    def fused():
        B.check(_native.lib().bs_crmsd_all_vs_all_row_stats_device(
            ctx.handle, vp(d_xyz.data_ptr()), n, L, gram, vp(d_out.data_ptr()), vp(d_lo2.data_ptr()),
            vp(d_hi2.data_ptr())))

    # alternating rounds, medians: the clock drifts over a run
    av_r, fu_r = [], []
    for _ in range(3):
        av_r.append(stream_ms(torch, ctx, avsa, 5)[0])
        fu_r.append(stream_ms(torch, ctx, fused, 5)[0])
    av_ms, fu_ms = float(np.median(av_r)), float(np.median(fu_r))
    row_stats()
    ctx.synchronize()
    fused_same = bool(torch.equal(d_lo.view(torch.int32), d_lo2.view(torch.int32))
                      and torch.equal(d_hi.view(torch.int32), d_hi2.view(torch.int32)))
    log(f"row stats in the epilogue: {fu_ms:.3f} ms with the all-vs-all ({av_ms:.3f} ms alone), "
        f"bit-identical {fused_same}")
    del d_lo2, d_hi2
    cn = min(n, args.cluster_n)
    d_tri = d_out
    if cn < n:  # the packed triangle of the leading cn x cn block
        ii = np.concatenate([i * n - i * (i + 1) // 2 + (np.arange(i + 1, cn) - i - 1) for i in range(cn)])
        d_tri = d_out[torch.from_numpy(ii).to(dev)].contiguous()
        torch.cuda.synchronize()
    m_i = np.zeros(cn, np.uint32)
    m_j = np.zeros(cn, np.uint32)
    m_d = np.zeros(cn, np.float32)
    t0 = time.perf_counter()
    B.check(_native.lib().bs_hierarchical_clustering_device(ctx.handle, vp(d_tri.data_ptr()), cn,
                                                             C.LINKAGES.index("average"),
                                                             m_i.ctypes.data_as(_native.c_u32p),
                                                             m_j.ctypes.data_as(_native.c_u32p),
                                                             m_d.ctypes.data_as(_native.c_fp)))
    cl_ms = (time.perf_counter() - t0) * 1e3
    # what the loop cannot do without: the triangle once, and per merge two rows read and one written
    alg_bytes = cn * (cn - 1) // 2 * 4 + sum(3 * k * 4 for k in range(2, cn + 1))
    # like for like at a CPU-sized sample: the first 1000 elements
    sn = 1000
    sub = d_out.cpu().numpy()
    idx = np.concatenate([i * n - i * (i + 1) // 2 + (np.arange(i + 1, sn) - i - 1) for i in range(sn)])
    up_s = np.ascontiguousarray(sub[idx])
    # both sides produce the merge list (the tree is rebuilt from it host-side
    # by the same code for either, outside the timed region)
    s_i = np.zeros(sn, np.uint32)
    s_j = np.zeros(sn, np.uint32)
    s_d = np.zeros(sn, np.float32)
    B.check(_native.lib().bs_hierarchical_clustering(ctx.handle, up_s.ctypes.data_as(_native.c_fp), sn,
                                                      C.LINKAGES.index("average"),
                                                      s_i.ctypes.data_as(_native.c_u32p),
                                                      s_j.ctypes.data_as(_native.c_u32p),
                                                      s_d.ctypes.data_as(_native.c_fp)))
    t0 = time.perf_counter()
    for _ in range(3):
        B.check(_native.lib().bs_hierarchical_clustering(ctx.handle, up_s.ctypes.data_as(_native.c_fp), sn,
                                                          C.LINKAGES.index("average"),
                                                          s_i.ctypes.data_as(_native.c_u32p),
                                                          s_j.ctypes.data_as(_native.c_u32p),
                                                          s_d.ctypes.data_as(_native.c_fp)))
    g_ms = (time.perf_counter() - t0) * 1e3 / 3
    t0 = time.perf_counter()
    oi, oj, od = O.hclust(up_s, sn, "average")
    c_ms = (time.perf_counter() - t0) * 1e3
    same = (np.array_equal(s_i[:sn - 1], oi) and np.array_equal(s_j[:sn - 1], oj)
            and np.array_equal(s_d[:sn - 1].view(np.uint32), np.asarray(od, np.float32).view(np.uint32)))
    log(f"clustering {cn}: {cl_ms:.1f} ms; row stats {rs_ms:.3f} ms; sample {sn}: gpu {g_ms:.1f} ms, cpu {c_ms:.1f} ms")
    out["clustering"] = {
        "workload": f"average-linkage agglomerative clustering of the {cn} x {cn} f32 triangle in HBM "
                    "(bs_hierarchical_clustering_device, merge order of the reference)",
        "n": cn,
        "ms": round(cl_ms, 2),
        "roofline": {"bound": "latency", "achieved": round(alg_bytes / (cl_ms * 1e-3) / 1e9, 1), "peak": 8000.0,
                     "unit": "GB/s", "frac": round(alg_bytes / (cl_ms * 1e-3) / 8e12, 4),
                     "traffic": None, "algorithmic_bytes": alg_bytes,
                     "note": "the triangle once, and per merge two rows read and one written; the time is the "
                             "chain of merges, each waiting for the one before"},
        "sample_1000": {"gpu_ms": round(g_ms, 2), "cpu_ms": round(c_ms, 2), "same_merges": bool(same),
                        "note": "bs_hierarchical_clustering (host triangle in, merge list out) against the "
                                "oracle's merge list; bit-identical merges, heights compared as f32 bits"},
        "cpu_baseline": {"value": round(c_ms, 2), "unit": "ms", "cores": 1, "kind": "port",
                         "sample": "oracle or_hclust (C restatement of hierarchical.rs:22-80) on the first "
                                   "1000 elements of the same matrix"},
        "row_stats_ms": round(rs_ms, 4),
        "row_stats_host_ms": round(rs_host_ms, 4),
        "row_stats_roofline": {"bound": "hbm", "achieved": round(tri_bytes / (rs_ms * 1e-3) / 1e9, 1),
                               "peak": 8000.0, "unit": "GB/s",
                               "frac": round(tri_bytes / (rs_ms * 1e-3) / 8e12, 4), "traffic": None},
        "row_stats_fused": {"workload": "the headline all-vs-all with its row minima and maxima taken in the "
                                        "Gram epilogue (bs_crmsd_all_vs_all_row_stats_device)",
                            "ms": round(fu_ms, 4), "all_vs_all_alone_ms": round(av_ms, 4),
                            "separate_calls_ms": round(av_ms + rs_ms, 4),
                            "bit_identical_to_separate": fused_same},
    }
    del d_lo, d_hi
    # ---- superposition of every conformation onto conformation 0 (FP64)
    d_rot = torch.empty((n, 9), dtype=torch.float64, device=dev)
    d_tr = torch.empty((n, 3), dtype=torch.float64, device=dev)
    d_rm = torch.empty(n, dtype=torch.float64, device=dev)
    d_sp = torch.empty_like(d_xyz)

    def sup():
        B.superpose_ensemble_device(d_xyz.data_ptr(), n, L, None, 0, d_rot.data_ptr(), d_tr.data_ptr(),
                                    d_rm.data_ptr(), d_sp.data_ptr(), ctx=ctx)

    sp_ms, sp_host_ms = stream_ms(torch, ctx, sup, reps)
    algo = n * L * 24 * 2  # coordinates read once, superposed coordinates written once
    rm = d_rm.cpu().numpy()
    k = 300
    t0 = time.perf_counter()
    want = np.array([O.superpose(x[0], x[m])[2] for m in range(k)])
    c_s = time.perf_counter() - t0
    out["superposition"] = {
        "workload": f"{n} x {L} ensemble fitted onto conformation 0: R, t, RMSD and the superposed "
                    "coordinates, FP64, in HBM (bs_superpose_ensemble_device)",
        "ms": round(sp_ms, 4),
        "host_ms": round(sp_host_ms, 4),
        "value": round(n / (sp_ms * 1e-3), 1),
        "unit": "conformations/s",
        "roofline": {"bound": "hbm", "achieved": round(algo / (sp_ms * 1e-3) / 1e9, 1), "peak": 8000.0,
                     "unit": "GB/s", "frac": round(algo / (sp_ms * 1e-3) / 8e12, 4), "traffic": None},
        "max_abs_rmsd_diff_vs_oracle": float(np.abs(rm[:k] - want).max()),
        "cpu_baseline": {"value": round(k / c_s, 1), "unit": "conformations/s", "cores": 1, "kind": "port",
                         "sample": f"oracle or_superpose on conformations 0..{k - 1}"},
    }
    del d_rot, d_tr, d_rm, d_sp
    log(f"superposition: {sp_ms:.3f} ms")
    # ---- ingestion: multi-model mmCIF -> CA ensemble
    text = synthetic_cif(args.ingest_models)
    B.Ensemble.from_text(text, select="ca", n_threads=16)  # warm the page cache and allocator
    t0 = time.perf_counter()
    e = B.Ensemble.from_text(text, select="ca", n_threads=16)
    in_s = time.perf_counter() - t0
    t0 = time.perf_counter()
    e1 = B.Ensemble.from_text(text, select="ca", n_threads=1)
    in1_s = time.perf_counter() - t0
    small = synthetic_cif(20)
    t0 = time.perf_counter()
    o = I.ensemble(small, selection="ca")
    o_s = time.perf_counter() - t0
    ok = bool(np.array_equal(e.xyz, e1.xyz) and np.array_equal(B.Ensemble.from_text(small, select="ca").xyz, o.xyz))
    out["ingestion"] = {
        "workload": f"mmCIF text of {args.ingest_models} models x 255 atoms ({len(text) / 1e6:.1f} MB), "
                    "CA selection -> (models, 15, 3) f64 (bs_ensemble_parse)",
        "ms": round(in_s * 1e3, 2),
        "value": round(len(text) / in_s / 1e6, 1),
        "unit": "MB/s",
        "threads": 16,
        "single_thread_MBps": round(len(text) / in1_s / 1e6, 1),
        "matches_oracle": ok,
        "cpu_baseline": {"value": round(len(small) / o_s / 1e6, 2), "unit": "MB/s", "cores": 1, "kind": "port",
                         "sample": f"oracle (Python restatement of the reference loader) on 20 models "
                                   f"({len(small) / 1e6:.2f} MB) of the same text"},
    }
    log(f"ingestion: {len(text) / in_s / 1e6:.0f} MB/s")
    # ---- clust TSV writer on the first 2000 elements
    tn = 2000
    idx = np.concatenate([i * n - i * (i + 1) // 2 + (np.arange(i + 1, tn) - i - 1) for i in range(tn)])
    m = B.RmsdMatrix(tn, np.ascontiguousarray(sub[idx]))
    import tempfile

    with tempfile.TemporaryDirectory() as td:
        pth = os.path.join(td, "d.tsv")
        C.write_tsv(m, pth, n_threads=16)
        t0 = time.perf_counter()
        C.write_tsv(m, pth, n_threads=16)
        w_s = time.perf_counter() - t0
        size = os.path.getsize(pth)
        t0 = time.perf_counter()
        C.write_tsv(m, pth, n_threads=1)
        w1_s = time.perf_counter() - t0
    out["tsv"] = {
        "workload": f"clust TSV of the {tn}-element sub-matrix ({tn * (tn - 1) // 2} lines, {size / 1e6:.1f} MB), "
                    "shortest round-trip f32 text (bs_write_distance_tsv)",
        "ms": round(w_s * 1e3, 2),
        "value": round(tn * (tn - 1) // 2 / w_s, 1),
        "unit": "lines/s",
        "threads": 16,
        "cpu_baseline": {"value": round(tn * (tn - 1) // 2 / w1_s, 1), "unit": "lines/s", "cores": 1,
                         "kind": "port", "sample": "the same writer on one thread (the oracle has no writer)"},
    }
    log(f"tsv: {w_s * 1e3:.1f} ms")
    return out


def host_info() -> dict:
    """The host the CPU baseline runs on: logical CPUs (nproc), the CPUs this
    process may run on (its affinity mask), the thread share the machine's
    environment grants (OMP_NUM_THREADS, where set), and lscpu's model,
    sockets, cores per socket and threads per core."""
    import subprocess

    info = {"nproc": os.cpu_count(), "affinity_cpus": len(os.sched_getaffinity(0)),
            "omp_num_threads": int(os.environ["OMP_NUM_THREADS"]) if os.environ.get("OMP_NUM_THREADS", "").isdigit()
            else None}
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        keys = {"Model name": "model", "Socket(s)": "sockets", "Core(s) per socket": "cores_per_socket",
                "Thread(s) per core": "threads_per_core"}
        for line in out.splitlines():
            k, _, v = line.partition(":")
            if k.strip() in keys:
                v = v.strip()
                info[keys[k.strip()]] = int(v) if v.isdigit() else v
    except (OSError, subprocess.SubprocessError):
        pass
    return info


def cpu_threads_default() -> int:
    """Every CPU this process may use, capped by the thread share the
    environment grants (OMP_NUM_THREADS) where one is set."""
    n = len(os.sched_getaffinity(0))
    omp = os.environ.get("OMP_NUM_THREADS", "")
    return min(n, int(omp)) if omp.isdigit() and int(omp) > 0 else n


def cpu_baseline(x: np.ndarray, target_s: float, threads: int) -> dict:
    """Times the FP64 oracle on rows [0, R) with R sized for ~target_s seconds."""
    from oracle import oracle as O

    n = x.shape[0]
    probe = min(n, 64)
    t0 = time.perf_counter()
    O.all_vs_all_rows(x, 0, probe, nthreads=threads)
    dt = time.perf_counter() - t0
    probe_pairs = sum(n - 1 - i for i in range(probe))
    rate = probe_pairs / max(dt, 1e-6)
    want_pairs = rate * target_s
    R, pairs = 0, 0
    while R < n and pairs + (n - 1 - R) <= want_pairs:
        pairs += n - 1 - R
        R += 1
    R = max(R, 8)
    pairs = sum(n - 1 - i for i in range(R))
    t0 = time.perf_counter()
    rows = O.all_vs_all_rows(x, 0, R, nthreads=threads)
    dt = time.perf_counter() - t0
    return {"rows": rows, "R": R, "pairs": pairs, "seconds": dt, "value": pairs / dt}


def main() -> None:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--n-conf", type=int, default=10000)
    ap.add_argument("--n-atoms", type=int, default=300)
    ap.add_argument("--plain-steps", type=int, default=3)
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--cpu-threads", type=int, default=0,
                    help="threads of the CPU baseline (0: every CPU of the affinity mask, capped by "
                         "OMP_NUM_THREADS where set)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-plain", action="store_true")
    ap.add_argument("--no-batch", action="store_true")
    ap.add_argument("--no-serving", action="store_true")
    ap.add_argument("--batch-ensembles", type=int, default=512)
    ap.add_argument("--serve-library", type=int, default=25000)
    ap.add_argument("--serve-qps", type=float, default=1000.0)
    ap.add_argument("--serve-requests", type=int, default=3000)
    ap.add_argument("--no-host-io", action="store_true", help="skip the host-buffer (PCIe-inclusive) calls")
    ap.add_argument("--no-next", action="store_true", help="skip the clustering / superposition / "
                    "ingestion / TSV leg")
    ap.add_argument("--cluster-n", type=int, default=10000)
    ap.add_argument("--ingest-models", type=int, default=2000)
    ap.add_argument("--calibrate-copy-mib", type=int, default=0,
                    help="copy a device buffer of this size once before the warmup (the "
                         "known-size kernel that scales rocprofv3 FETCH_SIZE / WRITE_SIZE)")
    args = ap.parse_args()

    if args.cpu_threads <= 0:
        args.cpu_threads = cpu_threads_default()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU only: the all-vs-all path runs on a single MI355X "
              "(multi-GPU sharding is a design note, not part of this build)", file=sys.stderr)
        sys.exit(2)

    import torch

    import bioshell_amd as B

    n, L = args.n_conf, args.n_atoms
    pairs = n * (n - 1) // 2
    log(f"generating {n} x {L} ensemble")
    x = B.generate_ensemble(20260, n, L, sigma=(0.5, 4.0), near_fraction=0.05, near_sigma=0.01)
    dev = torch.device("cuda:0")
    d_xyz = torch.from_numpy(x).to(dev)
    d_out = torch.empty(pairs, dtype=torch.float32, device=dev)
    d_plain = torch.empty(pairs, dtype=torch.float32, device=dev)
    torch.cuda.synchronize()
    if args.calibrate_copy_mib > 0:
        src = torch.ones(args.calibrate_copy_mib << 18, dtype=torch.float32, device=dev)
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
    ctx = B.Context(0)

    def step(method, out):
        B.crmsd_all_vs_all_device(d_xyz.data_ptr(), n, L, out.data_ptr(), method, ctx=ctx)

    # ---------------------------------------------------------- headline: BF16x3 Gram
    log("warmup")
    for _ in range(args.warmup):
        step(B.Method.BF16X3_GRAM, d_out)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step(B.Method.BF16X3_GRAM, d_out)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    # per-step device times, as the library's kernels stamp them
    hist = ctx.history(args.steps)
    main_ms = [h["main_ms"] for h in hist]
    prep_ms = [h["prep_ms"] for h in hist]
    fb_ms = [h["fallback_ms"] for h in hist]
    flagged = [h["flagged_pairs"] for h in hist]
    ms_per_step = dt * 1e3 / args.steps
    value = pairs / (dt / args.steps)
    log(f"bf16x3 gram: {ms_per_step:.3f} ms/step, kernel {np.mean(main_ms):.3f} ms")

    # ---------------------------------------------------------- plain per-pair kernel
    plain = None
    if not args.no_plain:
        step(B.Method.FP32_PLAIN, d_plain)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.plain_steps):
            step(B.Method.FP32_PLAIN, d_plain)
        torch.cuda.synchronize()
        plain_dt = (time.perf_counter() - t0) / args.plain_steps
        plain_kernel = [h["main_ms"] for h in ctx.history(args.plain_steps)]
        pk_ms = float(np.mean(plain_kernel))
        pk_tf = 18.0 * L * pairs / (pk_ms * 1e-3) / 1e12
        plain = {
            "method": "FP32_PLAIN",
            "value": round(pairs / plain_dt, 1),
            "ms_per_step": round(plain_dt * 1e3, 3),
            "kernel_ms": round(pk_ms, 3),
            "kernel": "plain_kernel<float, 4> (4 x 4 pairs per thread: centring, covariance, QCP, sqrt per pair)",
            "roofline": {
                "bound": "fp32_valu", "achieved": round(pk_tf, 2), "peak": PEAK_FP32_VALU_TFLOPS,
                "unit": "TFLOP/s", "frac": round(pk_tf / PEAK_FP32_VALU_TFLOPS, 4),
                "note": "algorithmic 18 L flops per pair (the covariance) over the kernel time; the peak "
                        "counts packed FP32, which this build does not emit, so half of it is the "
                        "ceiling for these FMAs",
            },
        }
        log(f"fp32 plain: {plain_dt * 1e3:.3f} ms/step")

    # ---------------------------------------------------------- host buffers in and out
    # (PCIe and staging included; never the headline value)
    host_io = None
    if not args.no_host_io:
        t0 = time.perf_counter()
        B.crmsd_all_vs_all(x, B.Method.BF16X3_GRAM, ctx=ctx)
        host_one_shot = time.perf_counter() - t0
        t0 = time.perf_counter()
        B.crmsd_all_vs_all_streamed(x, B.Method.BF16X3_GRAM, tile=4096, ctx=ctx)
        host_streamed = time.perf_counter() - t0
        log(f"host i/o: one-shot {host_one_shot * 1e3:.1f} ms, streamed 4096^2 {host_streamed * 1e3:.1f} ms")
        host_io = {
            "one_shot_ms": round(host_one_shot * 1e3, 2),
            "streamed_4096_ms": round(host_streamed * 1e3, 2),
            "streamed_pairs_per_s": round(pairs / host_streamed, 1),
            "note": "host f64 coordinates in, host f32 packed triangle out (72 MB H2D, 200 MB D2H)",
        }

    # ---------------------------------------------------------- roofline of the Gram kernel
    kernel_ms = float(np.mean(main_ms))
    algo_flops = 18.0 * L * pairs  # 9 L multiply-adds of the 3x3 covariance per pair
    achieved = algo_flops / (kernel_ms * 1e-3) / 1e12
    roofline = {
        "bound": "mfma",
        "achieved": round(achieved, 2),
        "peak": PEAK_BF16_TFLOPS,
        "unit": "TFLOP/s",
        "frac": round(achieved / PEAK_BF16_TFLOPS, 4),
        "traffic": traffic_bytes(n, L),
        "kernel": "gram_kernel<BF16x3>",
        "kernel_ms": round(kernel_ms, 4),
        "issued_mfma_tflops": round(3 * achieved, 2),
    }
    # the FP64 QCP epilogue inside the same kernel, as its own fraction
    fp64_per_pair = pmc_figure(n, L, "fp64_flops_per_pair")
    if fp64_per_pair is not None:
        f64 = fp64_per_pair * pairs / (kernel_ms * 1e-3) / 1e12
        roofline["fp64_epilogue"] = {
            "bound": "fp64_valu", "achieved": round(f64, 2), "peak": PEAK_FP64_VALU_TFLOPS,
            "unit": "TFLOP/s", "frac": round(f64 / PEAK_FP64_VALU_TFLOPS, 4),
            "flops_per_pair": fp64_per_pair,
            "source": "SQ_INSTS_VALU_{ADD,MUL,FMA,TRANS}_F64 of the Gram launch (FMA = 2 flops), "
                      "profiles/gram_bf16x3_10k_300_pmc.txt",
        }
    peaks = measured_peaks()
    if peaks.get("bf16_mfma_tflops"):
        peaks["gram_frac_of_measured_bf16"] = round(achieved / peaks["bf16_mfma_tflops"], 4)
    roofline["measured_peaks"] = peaks

    # ---------------------------------------------------------- error and CPU baseline
    err = None
    cpu = None
    if not args.no_cpu:
        log("cpu baseline")
        cb = cpu_baseline(x, args.cpu_seconds, args.cpu_threads)
        R = cb["R"]
        got = d_out.cpu().numpy()
        got_plain = d_plain.cpu().numpy() if plain else None
        ref_rows = cb["rows"]
        idx, want = [], []
        for i in range(R):
            j = np.arange(i + 1, n)
            idx.append(i * n - i * (i + 1) // 2 + (j - i - 1))
            want.append(ref_rows[i, i + 1:])
        idx = np.concatenate(idx)
        want = np.concatenate(want)
        e = np.abs(got[idx].astype(np.float64) - want)
        err = {
            "sample_pairs": int(idx.size),
            "bf16x3_max_abs": float(e.max()),
            "bf16x3_mean_abs": float(e.mean()),
        }
        if plain:
            ep = np.abs(got_plain[idx].astype(np.float64) - want)
            err["fp32_plain_max_abs"] = float(ep.max())
            err["fp32_plain_mean_abs"] = float(ep.mean())
        cpu = {
            "value": round(cb["value"], 1),
            "unit": "superpositions/s",
            "cores": args.cpu_threads,
            "host": host_info(),
            "kind": "port",
            "sample": f"rows 0..{R - 1} of the same 10,000 x 300 ensemble ({cb['pairs']} pairs), "
                      f"FP64 QCP oracle, {cb['seconds']:.1f} s",
        }
        one = cpu_baseline(x, args.cpu_seconds / 2, 1)  # the same oracle on one thread
        cpu["one_thread"] = {
            "value": round(one["value"], 1),
            "cores": 1,
            "sample": f"rows 0..{one['R'] - 1} ({one['pairs']} pairs), {one['seconds']:.1f} s",
        }

    nxt = None if args.no_next else next_rows_leg(args, B, torch, log, ctx, d_xyz, d_out, x)
    batch = None if args.no_batch else batch_leg(args, B, torch, log)
    serving = None if args.no_serving else serving_leg(args, B, log)

    out = {
        "metric": METRIC,
        "value": round(value, 1),
        "unit": "superpositions/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded NeRF random-walk chains + Gaussian noise + random rigid motion)",
        "config": {
            "workload": f"all-vs-all crmsd, {n} conformations x {L} CA atoms, 5% near-identical "
                        f"(sigma 0.01 A), others sigma U(0.5,4) A; packed f32 triangle in HBM",
            "n_conf": n,
            "n_atoms": L,
            "pairs": pairs,
            "method": "BF16X3_GRAM (bf16 hi/lo MFMA, fp32 accumulation, fp64 QCP epilogue + fp64 re-evaluation)",
        },
        "stages_ms": {
            "prep": round(float(np.mean(prep_ms)), 4),
            "gram": round(kernel_ms, 4),
            "fallback": round(float(np.mean(fb_ms)), 4),
        },
        "flagged_pairs": int(np.mean(flagged)),
        "host_io": host_io,
        "plain_gpu": plain,
        "speedup_vs_plain": round(value / plain["value"], 2) if plain else None,
        "error_vs_fp64": err,
        "roofline": roofline,
        "cpu_baseline": cpu,
        "batch": batch,
        "serving": serving,
        "next": nxt,
    }
    print(json.dumps(out), flush=True)
    ctx.close()


if __name__ == "__main__":
    main()
