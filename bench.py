#!/usr/bin/env python3
"""Benchmark of the GLIDE hot path on one MI355X: index build seconds + graph recall@32, search QPS.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload cfg1|cfg1-navigable|cfg0|cfg2|cfg3|cfg4] [--no-cpu] [--headline-only]

A "step" is one beam-search pass of the whole query batch (10 000 queries, top-10) over the finished index.
Before the timed steps the index is built once on the GPU (partition -> NN-descent -> sub-graph build + boundary
merge -> reverse edges -> refine) and its stage times, the kNN-graph recall@32 against exact neighbours and the
recall@10 of the whole beam sweep (32 ... 512, the reference's range) are measured.  Stdout carries one
`{"bench_detail": <workload>, ...}` JSON line per workload measured (the medium configuration cfg1 first, then the same
shapes on navigable data and the other single-GPU configurations cfg0, cfg2, cfg3: build stages, graph recall, beam
sweep, stage rooflines, roofline of the timed search kernel, the CPU restatement's recall and throughput at the same
beam) and ends with ONE compact line of a few KB: the benchmark record of cfg1 (`headline()` below).  The same details
go to the file --details-file names.  cfg4 (50M rows staged from pinned host memory) has a run of its own: --workload cfg4.

Everything on the product path goes through libglide_hip.so.  torch is imported only to compute exact ground
truth on the GPU (a checker); the CPU oracle is used only for the cpu_baseline legs.
"""
import argparse
import json
import os
import re
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
MFMA_F32_PEAK_TFLOPS = 157.3
SWEEP_BEAMS = (32, 64, 128, 256, 512)       # the reference accepts beams up to 512 (kernel_config.cuh:41-60)
NAMED_BEAMS = {"cfg1": (32, 64, 128, 256)}  # the medium configuration names its beams; 512 is swept there as an extra
TRAFFIC_PROFILE = os.path.join(ROOT, "profiles", "search_kernels_hbm_traffic.md")
VALU_PROFILE = os.path.join(ROOT, "profiles", "build_refine_kernels_counters.md")
NND_PROFILE = os.path.join(ROOT, "profiles", "nnd_kernels_cfg1_rounds_and_counters.md")
GATHER_PROFILE = os.path.join(ROOT, "profiles", "gather_probe_scattered_rows.md")
NND_OFFERS_NOTE = ("nnd_offers: distinct offers the merge steps found in the offer tables, all rounds.  nnd_offers_declined_by_threshold: offers a "
                   "join did not send because their distance was not below the threshold their target announced (the distance of its 64th "
                   "best offer of the round before, announced only by nodes whose table was five eighths full).  Nothing depends on the order "
                   "of arrival: two builds with one seed give the same graph (tests/test_gpu_nnd.py::test_nnd_same_seed_same_graph).")


def measured_traffic(workload, beam):
    """HBM bytes one launch of the timed search kernel moves, from the committed counter summary: two `rocprofv3 --pmc` runs
    of this script (FETCH_SIZE, then WRITE_SIZE, KiB per dispatch), each scaled by what the same counter reads for the
    plain copy kernel of known size (--copy-calibration).  The table rows are `| workload | beam | FETCH_SIZE KiB |
    WRITE_SIZE KiB | fetch scale | write scale |`.  A (workload, beam) the file does not hold reports null: the value is
    an offline measurement, tied to the commit the file names, not something this run derives."""
    try:
        text = open(TRAFFIC_PROFILE).read()
    except OSError:
        return None
    for m in re.finditer(r"^\|\s*([\w-]+)\s*\|\s*(\d+)\s*\|\s*([\d.]+)\s*\|\s*([\d.]+)\s*\|\s*([\d.]+)\s*\|\s*([\d.]+)\s*\|", text, re.M):
        if m.group(1) == workload and int(m.group(2)) == beam:
            return dict(bytes=float(m.group(3)) * 1024 * float(m.group(5)) + float(m.group(4)) * 1024 * float(m.group(6)),
                        source="profiles/" + os.path.basename(TRAFFIC_PROFILE))
    return None


def scattered_row_ceiling(row_bytes):
    """The rate (GB/s) at which this GPU reads rows of `row_bytes` scattered over a table when a kernel does nothing else,
    from the committed summary of `--gather-calibration` (the probe kernel's best figure over its residencies): what the
    search kernels' row gathers can reach at all, below the 8 TB/s the HBM stacks are specified at.  The table rows are
    `| row bytes | best GB/s | fraction of 8 TB/s |`; the row of the nearest length at or above `row_bytes` is used."""
    try:
        text = open(GATHER_PROFILE).read()
    except OSError:
        return None
    rows = sorted((int(m.group(1)), float(m.group(2))) for m in re.finditer(r"^\|\s*(\d+)\s*\|\s*([\d.]+)\s*\|\s*[\d.]+\s*\|\s*$", text, re.M))
    for length, gbs in rows:
        if length >= row_bytes:
            return dict(row_bytes=length, GBps=gbs, source="profiles/" + os.path.basename(GATHER_PROFILE))
    return dict(row_bytes=rows[-1][0], GBps=rows[-1][1], source="profiles/" + os.path.basename(GATHER_PROFILE)) if rows else None


def measured_stage(stage, workload):
    """(vector-ALU wave instructions, FETCH_SIZE KiB, vector-ALU yardstick in G wave instructions / s, fetch scale) of one
    build stage (all launches of `build_kernel`, or the launch of `refine_kernel`) on one workload, from the committed
    counter summary: SQ_INSTS_VALU and FETCH_SIZE per launch from `rocprofv3 --pmc` runs of this script, the yardstick
    from --valu-calibration (compare + select), the scale from --copy-calibration.  The builds are reproducible, so the
    counts belong to the workload, not to a run.  None for a pair the file does not hold."""
    try:
        text = open(VALU_PROFILE).read()
    except OSError:
        return None
    for m in re.finditer(r"^\|\s*([\w+]+)\s*\|\s*([\w-]+)\s*\|\s*(\d+)\s*\|\s*(\d+)\s*\|\s*([\d.]+)\s*\|\s*([\d.]+)\s*\|\s*$", text, re.M):
        if m.group(1) == stage and m.group(2) == workload:
            return float(m.group(3)), float(m.group(4)), float(m.group(5)), float(m.group(6))
    return None


def measured_knn(workload):
    """(atomic lane operations issued by pairs of adjacent lanes on one line, issued by single lanes, yardstick rates of the
    two in G/s) of the NN-descent stage of one workload, from the committed counter summary: TCP_TCC_ATOMIC_*_REQ summed
    over the launches of a build (`rocprofv3 --pmc` run of this script), the rates from --atomic-calibration.  The build
    is reproducible, so the counts belong to the workload.  None for a workload the file does not hold."""
    try:
        text = open(NND_PROFILE).read()
    except OSError:
        return None
    for m in re.finditer(r"^\|\s*knn\s*\|\s*([\w-]+)\s*\|\s*(\d+)\s*\|\s*(\d+)\s*\|\s*([\d.]+)\s*\|\s*([\d.]+)\s*\|\s*$", text, re.M):
        if m.group(1) == workload:
            return float(m.group(2)), float(m.group(3)), float(m.group(4)), float(m.group(5))
    return None


def search_kernel_name(dim, degree, beam, queries, compute_units, of_bytes=False):
    """The kernel glide_hip_search launches for this shape, as a profiler names it (search.hip: launch_search).  of_bytes: rows and
    queries are whole numbers 0..255 and searched as bytes (a second launch finds no query left over)."""
    shape = "%d, %d, %d" % (64 if degree <= 64 else 128 if degree <= 128 else 256,
                            64 if beam <= 64 else 128 if beam <= 128 else 256 if beam <= 256 else 512,
                            (-1 if dim <= 128 else -2) if of_bytes else 1 if dim <= 128 else 2 if dim <= 256 else 4 if dim <= 512 else 8 if dim <= 1024 else 16)
    whole = "true" if beam == 512 else "false"      # the whole of the widest beam: merged in the registers
    if dim > 256 and queries * 4 <= 2 * 4 * compute_units:
        return "search_team_kernel<%s, %s>" % (shape, whole)
    return "search_kernel<%s, %s, false>" % (shape, whole)


def measured_knn_bytes(workload):
    """HBM bytes (read + written) of all launches of the NN-descent stage of one workload, from the committed counter
    summary: FETCH_SIZE and WRITE_SIZE summed over the stage's launches, each scaled by the copy kernel's reading.  The
    table row is `| knn-hbm | workload | FETCH_SIZE KiB | WRITE_SIZE KiB | fetch scale | write scale |`."""
    try:
        text = open(NND_PROFILE).read()
    except OSError:
        return None
    for m in re.finditer(r"^\|\s*knn-hbm\s*\|\s*([\w-]+)\s*\|\s*(\d+)\s*\|\s*(\d+)\s*\|\s*([\d.]+)\s*\|\s*([\d.]+)\s*\|\s*$", text, re.M):
        if m.group(1) == workload:
            return float(m.group(2)) * 1024 * float(m.group(4)) + float(m.group(3)) * 1024 * float(m.group(5))
    return None


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="cfg1", choices=["cfg0", "cfg1", "cfg1-navigable", "cfg2", "cfg3", "cfg4"])
    ap.add_argument("--headline-only", action="store_true", help="cfg1 only: skip the other configurations and the navigable variant")
    ap.add_argument("--cfg4-rows", type=int, default=50_000_000, help="rows of the cfg4 run (the named size is 50M)")
    ap.add_argument("--nnd-iterations", type=int, default=0)
    ap.add_argument("--no-cpu", action="store_true", help="skip the cpu_baseline leg")
    ap.add_argument("--knn-only", action="store_true", help="partition + NN-descent kNN graph of the workload only (for kernel profiles)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run the plain copy kernel on 1 GiB x steps (yardstick for rocprofv3 byte counters) and exit")
    ap.add_argument("--valu-calibration", action="store_true",
                    help="only run the register-only multiply-add kernel (yardstick for the vector-ALU issue rate) and exit")
    ap.add_argument("--atomic-calibration", action="store_true",
                    help="only run the scattered-atomics kernel (yardstick for the NN-descent offers and slot reservations) and exit")
    ap.add_argument("--gather-calibration", action="store_true",
                    help="only run the scattered-row read kernel (yardstick for the search kernels' row gathers) and exit")
    ap.add_argument("--details-file", default=os.path.join("gpurun_out", "bench_full.json"),
                    help="where the per-workload details are written as one JSON file (relative to the repository root)")
    ap.add_argument("--queries", type=int, default=0, help="use only the first N queries of the workload (small-batch measurements)")
    ap.add_argument("--extra-beams", default="", help="comma-separated beams to add to the sweep, e.g. 288,320,384,448,480")
    ap.add_argument("--partition-only", type=int, default=0, metavar="C",
                    help="only time partition assignment of 1M x 128 rows against C centroids (fp32 matrix-core tile) and exit")
    return ap.parse_args()


WORKLOADS = {
    # name: (num, partitions, knn degree, NN-descent iterations, queries, description, dim, metric, graph degree)
    "cfg0": (100_000, 10, 64, 8, 1_000, "cfg0: 100k x 128 fp32 clipped/rounded 64-component GMM, L2, degree 32, NN-descent k=64 x 8 iterations, 1k queries", 128, 0, 32),
    "cfg1": (1_000_000, 16, 32, 20, 10_000, "cfg1: 1M x 128 fp32 clipped/rounded 64-component GMM, L2, 16 partitions, degree 32, 10k queries top-10, beams 32/64/128/256", 128, 0, 32),
    "cfg1-navigable": (1_000_000, 16, 32, 20, 10_000, "cfg1 shapes on integer-valued data of low intrinsic dimension (12-d latent, 0..255): 1M x 128, 16 partitions, degree 32, 10k queries top-10", 128, 0, 32),
    "cfg2": (1_000_000, 16, 32, 20, 10_000, "cfg2: 1M x 96 fp32 L2-normalised 256-component GMM, cosine, 16 partitions, degree 32, 10k queries top-10", 96, 1, 32),
    "cfg3": (1_000_000, 16, 64, 20, 1_000, "cfg3: 1M x 960 fp32 Beta(0.5,2) x per-cluster scales, L2, 16 partitions, degree 64, 1k queries top-10", 960, 0, 64),
}


def make_data(workload, num, nq):
    import numpy as np
    from glide_amd import datasets as D
    if workload == "cfg1-navigable":
        return D.lowdim_integer(num, 128, seed=1234), D.lowdim_integer(nq, 128, seed=4321)
    if workload == "cfg2":
        return D.gmm_normalized(num, 96, seed=1234), D.gmm_normalized(nq, 96, seed=4321)
    if workload == "cfg3":
        return D.beta_scaled(num, 960, seed=1234), D.beta_scaled(nq, 960, seed=4321)
    return D.gmm_clipped(num, 128, seed=1234), D.gmm_clipped(nq, 128, seed=4321)


def exact_knn(torch, base, queries, k, exclude_self_offset=None, chunk=2048):
    """Exact top-k by brute force on the GPU (checker).  Integer-valued inputs below 2^24 make the norm trick exact."""
    b = torch.from_numpy(base).cuda()
    bn = (b * b).sum(1)
    out = []
    for s in range(0, queries.shape[0], chunk):
        q = torch.from_numpy(queries[s:s + chunk]).cuda()
        d = (q * q).sum(1, keepdim=True) + bn[None] - 2.0 * (q @ b.T)
        if exclude_self_offset is not None:
            idx = torch.arange(q.shape[0], device="cuda")
            d[idx, idx + s + exclude_self_offset] = float("inf")
        out.append(d.topk(k, largest=False).indices.cpu())
    return torch.cat(out).numpy()


def run_workload(args, workload, torch, want_cpu):
    import numpy as np
    from glide_amd import capi, datasets as D, index as G

    num, parts, knn_degree, nnd_iters, nq, desc, dim, metric, degree = WORKLOADS[workload]
    if args.nnd_iterations:
        nnd_iters = args.nnd_iterations
    top_k = 10
    info_cus = capi.device_info()["compute_units"]
    t0 = time.time()
    data, queries = make_data(workload, num, nq)
    if args.queries:
        nq = min(nq, args.queries)
        queries = np.ascontiguousarray(queries[:nq])
    gen_s = time.time() - t0

    d_data = capi.DeviceArray.from_numpy(data)
    res = {}
    pp = G.PartitionParameter(centroid_num=parts, boundary_factor=1.04, sample_factor=0.01, metric=metric)   # reference test.sh:10-12
    d_re, d_map, h_start, h_len, d_cent = G.preprocess(pp, d_data, res)
    nn = G.NNDescentParameter(graph_degree=knn_degree, max_iterations=nnd_iters)
    d_knn = G.build_nnd(nn, d_re, h_start, h_len, res, stats=True)

    # graph recall@k of the kNN graph inside each partition (what NN-descent is asked to find) on 500 nodes per partition
    knn = d_knn.numpy()
    rdata = d_re.numpy()
    h_map = d_map.numpy()
    k_eval = min(32, knn_degree)
    per_part, glob = [], []
    sample_global_ids, sample_rows = [], []
    for s, l in zip(h_start.tolist(), h_len.tolist()):
        if l <= 2 * knn_degree:
            continue
        m = min(500, l)
        sub = rdata[s:s + l]
        gt = exact_knn(torch, sub, sub[:m], k_eval, exclude_self_offset=0)
        per_part.append(D.recall(knn[s:s + m, :k_eval], gt, k_eval))
        if s < num:
            sample_global_ids.append(h_map[s:s + m])
            sample_rows.append((s, m))
    # the same nodes against exact neighbours over the whole data set (capped by partition locality)
    if sample_global_ids:
        gids = np.concatenate(sample_global_ids)
        b = torch.from_numpy(data).cuda()
        bn = (b * b).sum(1)
        q = b[torch.from_numpy(gids.astype(np.int64)).cuda()]
        d = (q * q).sum(1, keepdim=True) + bn[None] - 2.0 * (q @ b.T)
        d[torch.arange(q.shape[0], device="cuda"), torch.from_numpy(gids.astype(np.int64)).cuda()] = float("inf")
        gt_glob = d.topk(k_eval, largest=False).indices.cpu().numpy()
        found = np.concatenate([h_map[s + knn[s:s + m, :k_eval].astype(np.int64)] for s, m in sample_rows])
        glob.append(D.recall(found, gt_glob, k_eval))
        del b, bn, q, d
    graph_recall_partition = float(np.mean(per_part))
    graph_recall_global = float(glob[0]) if glob else None
    del rdata, knn

    index = G.GLIDE(degree, d_data, d_cent, metric)
    bp = G.IndexParameter(graph_degree=degree, knn_degree=knn_degree, relaxant_factor=1.05)   # test.sh:16
    sp_knn = G.make_search_parameter(64, knn_degree)         # test.sh:17 build beam
    sp_ref = G.make_search_parameter(128, knn_degree)        # test.sh:18 refine beam (hash sized with knn_degree, small_build.cu:76-82)
    index.build(bp, sp_knn, sp_ref, d_knn, h_start, h_len, d_map, d_re, res, counters=True)
    build_sec = res["pre_time"] + res["knn_time"] + res["index_time"] + res["refine_time"]
    graph = index.d_graph.numpy()
    d_bytes = index._byte_rows()       # rows of whole numbers 0..255 are searched as bytes, with the same ids and distances
    row_bytes = capi.byte_rows_bytes(1, dim) if d_bytes is not None else dim * 4
    holes = float((graph == 0xFFFFFFFF).mean())

    # ---- search sweep
    gt = exact_knn(torch, data, queries, top_k)
    d_q = capi.DeviceArray.from_numpy(queries)
    d_ids, d_dists = capi.DeviceArray((nq, top_k), np.uint32), capi.DeviceArray((nq, top_k), np.float32)
    sweep = []

    def measure(beam):
        sp = G.make_search_parameter(beam, degree, top_k)
        cnt = capi.new_counters()
        index.search(sp, d_q, counters=cnt, out=(d_ids, d_dists))
        capi.synchronize()
        c = capi.read_counters(cnt)
        r = {}
        index.search(sp, d_q, result=r, out=(d_ids, d_dists))
        rec = D.recall(d_ids.numpy(), gt, top_k)
        # algorithmic bytes of one launch: query rows + centroid table once + graph rows + scored data rows (as they are read) + results
        alg = nq * dim * 4 + parts * dim * 4 + int(c[2]) * degree * 4 + int(c[1]) * row_bytes + nq * top_k * 8
        sweep.append(dict(beam=beam, recall_at_10=rec, qps=r["QPS"], ms=r["search_time"] * 1e3, iterations_per_query=c[0] / nq,
                          rows_per_query=c[1] / nq, algorithmic_bytes=alg))
        return rec

    recalls = {beam: measure(beam) for beam in SWEEP_BEAMS}
    for beam in sorted({int(b) for b in args.extra_beams.split(",") if b} - set(SWEEP_BEAMS)):
        measure(beam)
    sweep.sort(key=lambda s: s["beam"])
    # "the smallest beam reaching the target": where a power of two reaches it and the one before does not, the three
    # beams between them (steps of an eighth of the larger one) are measured as well
    if workload not in NAMED_BEAMS:
        for lo, hi in zip(SWEEP_BEAMS, SWEEP_BEAMS[1:]):
            if recalls[lo] < 0.95 <= recalls[hi]:
                for beam in range(lo + (hi - lo) // 4, hi, (hi - lo) // 4):
                    measure(beam)
        sweep.sort(key=lambda s: s["beam"])
    # the metric's operating point: the smallest beam that reaches recall@10 0.95; where none does (see recall_target_met)
    # the widest beam of the reference's range is timed instead and the line says so
    named = [s for s in sweep if workload not in NAMED_BEAMS or s["beam"] in NAMED_BEAMS[workload]]
    ok = [s for s in named if s["recall_at_10"] >= 0.95]
    chosen = min(ok, key=lambda s: s["beam"]) if ok else named[-1]

    # ---- timed steps at the chosen beam: HIP events on the launch stream, warm-up first
    sp = G.make_search_parameter(chosen["beam"], degree, top_k)
    for _ in range(args.warmup):
        index.search(sp, d_q, out=(d_ids, d_dists))
    capi.synchronize()
    e0, e1 = capi.Event(), capi.Event()
    w0 = time.time()
    e0.record()
    for _ in range(args.steps):
        capi.search(index.d_data, num, dim, index.d_graph, degree, index.d_centroids, parts, index.d_start_points, d_q, nq, top_k,
                    sp.beam, sp.max_iterations, sp.min_iterations, sp.hash_bit, sp.hash_reset_interval, metric, d_ids, d_dists, byte_rows=d_bytes)
    e1.record()
    gpu_ms = e0.elapsed_ms(e1)
    capi.synchronize()
    wall_ms = (time.time() - w0) * 1e3
    ms_per_step = wall_ms / args.steps
    kernel_ms = gpu_ms / args.steps
    achieved = chosen["algorithmic_bytes"] / (kernel_ms * 1e-3) / 1e9

    # ---- the build kernels against their own rooflines: algorithmic bytes (from the kernels' counters: graph rows read
    # and data rows scored, prune rows included) or flops over the stage's GPU time
    det = {**res["pre_stages"], **res["build_stages"]}
    reorder_rows = int(h_len.sum())

    def hbm_stage(seconds, nbytes):
        gbs = nbytes / seconds / 1e9 if seconds > 0 else 0.0
        out = dict(bound="hbm", seconds=seconds, algorithmic_bytes=int(nbytes), achieved=gbs, peak=HBM_PEAK_GBS, unit="GB/s", frac=gbs / HBM_PEAK_GBS)
        return out

    def graph_stage(seconds, nbytes, stage):
        """`frac` is the fraction of the published HBM peak the stage's measured traffic (committed FETCH_SIZE counters) comes
        to.  The per-point graph kernels are bound by vector-ALU issue where their searches stay in cache (the sorting
        networks, cross-lane sums and distances of the beam loop): their instruction rate against the probe kernel's rate
        for compare + select pairs is reported beside it as `valu_yardstick_frac`, and the bytes their algorithm names,
        which a partition's cache may serve many times over, without a fraction."""
        out = dict(bound="hbm", seconds=seconds, algorithmic_bytes=int(nbytes), algorithmic_GBps=nbytes / seconds / 1e9 if seconds > 0 else 0.0,
                   peak=HBM_PEAK_GBS, unit="GB/s")
        m = measured_stage(stage, workload)
        if m and seconds > 0:
            instructions, fetch_kib, yardstick, scale = m
            valu, hbm = instructions / seconds / 1e9, fetch_kib * 1024 * scale / seconds / 1e9
            out.update(achieved=hbm, frac=hbm / HBM_PEAK_GBS, valu_G_wave_instructions_per_s=valu, valu_yardstick=yardstick,
                       valu_yardstick_frac=valu / yardstick, limited_by="valu" if valu / yardstick >= hbm / HBM_PEAK_GBS else "hbm",
                       source="profiles/" + os.path.basename(VALU_PROFILE))
        else:
            out.update(achieved=None, frac=None, note="no counters committed for this stage on this workload")
        return out

    # a row as the kernels of a stage read it; looked at in fp16 first: without the few that are then read in fp32 as well
    read = {k: {"bytes": row_bytes, "fp16 first": dim * 2, "fp32": dim * 4}[v] for k, v in res["rows_read"].items()}

    stage_rooflines = {}
    assign_flops = 2.0 * num * parts * dim
    a = hbm_stage(det["assign"], num * dim * 4 + num * 12)
    a_mfma = assign_flops / det["assign"] / 1e12 / MFMA_F32_PEAK_TFLOPS if det["assign"] > 0 else 0.0
    a.update(mfma_tflops=a_mfma * MFMA_F32_PEAK_TFLOPS, mfma_peak_tflops=MFMA_F32_PEAK_TFLOPS, hbm_frac=a["frac"], mfma_frac=a_mfma,
             frac=max(a["frac"], a_mfma), bound="hbm" if a["frac"] >= a_mfma else "mfma")
    stage_rooflines["assign"] = a
    stage_rooflines["reorder"] = hbm_stage(det["reorder"], (num + reorder_rows) * dim * 4)
    # NN-descent: `frac` is the stage's measured HBM traffic (committed FETCH_SIZE + WRITE_SIZE sums over its launches) over
    # its time against the published peak.  What holds its kernels is what a CU's memory pipeline charges per distinct
    # cache line, atomic operations above all: the time its atomics take at the rates of the probe kernel, as a fraction of
    # the stage, is `atomic_yardstick_frac`.
    mk, mb = measured_knn(workload), measured_knn_bytes(workload)
    if res["knn_time"] > 0 and (mk or mb):
        k = dict(bound="hbm", seconds=res["knn_time"], peak=HBM_PEAK_GBS, unit="GB/s", achieved=None, frac=None,
                 source="profiles/" + os.path.basename(NND_PROFILE))
        if mb:
            k.update(hbm_bytes=int(mb), achieved=mb / res["knn_time"] / 1e9, frac=mb / res["knn_time"] / 1e9 / HBM_PEAK_GBS)
            k["hbm_frac"] = k["frac"]
        if mk:
            paired, single, rate_pairs, rate_single = mk
            at_yardstick = paired / rate_pairs / 1e9 + single / rate_single / 1e9
            k.update(limited_by="scattered atomics", atomic_lane_operations_in_pairs=int(paired), atomic_lane_operations_single=int(single),
                     atomic_peak_pairs_G_per_s=rate_pairs, atomic_peak_single_G_per_s=rate_single,
                     seconds_at_the_atomic_yardstick_rates=at_yardstick, atomic_yardstick_frac=at_yardstick / res["knn_time"])
        stage_rooflines["knn"] = k
    if "build_counters" in res:
        _, rows, grows = res["build_counters"]
        stage_rooflines["subgraph+boundary"] = graph_stage(det["subgraph"] + det["boundary"],
                                                           reorder_rows * dim * 4 + grows * knn_degree * 4 + rows * read["subgraph"] + reorder_rows * degree * 4,
                                                           "subgraph+boundary")
    if "refine_counters" in res:
        _, rows, grows = res["refine_counters"]
        stage_rooflines["refine"] = graph_stage(det["refine"], num * dim * 4 + 2 * num * degree * 4 + grows * degree * 4 + rows * read["refine"], "refine")

    bound = D.reachable_recall_bound(graph, d_cent.numpy(), index.d_start_points.numpy(), queries, gt, metric)

    out = dict(
        workload=desc, rows_read=dict(res["rows_read"], search="bytes" if d_bytes is not None else "fp32"), gen_sec=gen_s, build_sec=build_sec, stage_rooflines=stage_rooflines,
        build_stages=dict(pre=res["pre_time"], knn=res["knn_time"], index=res["index_time"], refine=res["refine_time"],
                          detail={**res["pre_stages"], **res["build_stages"]}),
        nnd_iterations=nnd_iters, nnd_offers=res["nnd_stats"][0], nnd_offers_declined_by_threshold=res["nnd_stats"][1],
        nnd_offers_note=NND_OFFERS_NOTE,
        graph_recall_at_32=graph_recall_partition, graph_recall_at_32_global=graph_recall_global,
        partition_sizes=[int(x) for x in h_len], empty_slots_fraction=holes,
        sweep=sweep, beam=chosen["beam"], recall_at_10=chosen["recall_at_10"], recall_target_met=bool(ok),
        reachable_recall_bound=bound[0], reachable_fraction_of_points=bound[1],
        qps=nq * args.steps / (wall_ms * 1e-3), ms_per_step=ms_per_step, kernel_ms=kernel_ms,
        roofline=dict(bound="hbm", achieved=achieved, peak=HBM_PEAK_GBS, unit="GB/s", frac=achieved / HBM_PEAK_GBS,
                      traffic=(measured_traffic(workload, chosen["beam"]) or {}).get("bytes"),
                      traffic_source=(measured_traffic(workload, chosen["beam"]) or {}).get("source"),
                      kernel=search_kernel_name(dim, degree, chosen["beam"], nq, info_cus, d_bytes is not None),
                      algorithmic_bytes_per_launch=chosen["algorithmic_bytes"]),
    )
    # what scattered rows of this length can be read at on this GPU at all (a probe kernel that only gathers rows)
    ceiling = scattered_row_ceiling(row_bytes)
    if ceiling:
        out["roofline"].update(scattered_row_ceiling_GBps=ceiling["GBps"], scattered_row_ceiling_frac=ceiling["GBps"] / HBM_PEAK_GBS,
                               scattered_row_ceiling_source=ceiling["source"])
        # bytes that leave L2, as measured: the algorithmic ones count a row for every search that scores it
        if out["roofline"]["traffic"]:
            out["roofline"]["frac_of_scattered_row_ceiling"] = out["roofline"]["traffic"] / (kernel_ms * 1e6) / ceiling["GBps"]

    if want_cpu == "full":
        out["cpu_baseline"] = cpu_baseline(data, queries, graph, d_cent.numpy(), index.d_start_points.numpy(), sp, top_k, gt, metric)
    elif want_cpu:
        out["cpu_baseline"] = cpu_baseline(data, queries, graph, d_cent.numpy(), index.d_start_points.numpy(), sp, top_k, gt, metric,
                                           search_only=True, max_queries=500)
    return out


def cpu_baseline(data, queries, graph, centroids, start_points, sp, top_k, gt, metric=0, search_only=False, max_queries=10_000):
    """The CPU restatement of the reference algorithm, timed on this box's host cores on a bounded sample."""
    import numpy as np
    from glide_amd import datasets as D
    from oracle import oracle as O
    cores = os.cpu_count() or 1
    try:
        cores = len(os.sched_getaffinity(0))
    except Exception:
        pass
    cores = min(cores, int(os.environ.get("OMP_NUM_THREADS", cores)))
    nq = min(queries.shape[0], max_queries)
    t = time.time()
    ids, _, _ = O.search(data, graph, centroids, start_points, queries[:nq], top_k, sp.beam, sp.max_iterations, sp.min_iterations,
                         sp.hash_bit, sp.hash_reset_interval, metric, threads=cores)
    search_s = time.time() - t
    if search_only:
        return dict(value=nq / search_s, unit="queries/s", cores=cores, kind="port",
                    sample="beam search of the first %d queries (same index, beam %d) with the CPU restatement, %d threads" % (nq, sp.beam, cores),
                    recall_at_10=D.recall(ids, gt[:nq], top_k))
    # NN-descent build of one partition-sized sample (1M / 16 points) with the same degree / 10 iterations
    n_s = min(62_500, data.shape[0])
    t = time.time()
    O.nnd_build(data[:n_s], np.array([0], np.uint32), np.array([n_s], np.uint32), 32, 10, 0, threads=cores)
    nnd_s = time.time() - t
    t = time.time()
    n_bf = min(queries.shape[0], 1000)
    O.bruteforce_knn(data, queries[:n_bf], top_k, metric, threads=cores)
    bf_s = time.time() - t
    return dict(value=nq / search_s, unit="queries/s", cores=cores, kind="port",
                sample="beam search of the first %d queries (same index, beam %d) with the CPU restatement, %d threads" % (nq, sp.beam, cores),
                recall_at_10=D.recall(ids, gt[:nq], top_k),
                nnd_points_per_sec=n_s / nnd_s, nnd_sample="NN-descent k=32 x 10 iterations on the first %d points as one partition" % n_s,
                bruteforce_qps=n_bf / bf_s, bruteforce_sample="exact top-%d of the first %d queries over all %d rows" % (top_k, n_bf, data.shape[0]))


def main():
    args = parse()
    if args.gpus != 1:
        print("bench.py measures one GPU: this build has no multi-GPU path (--gpus %d refused)" % args.gpus, file=sys.stderr)
        sys.exit(2)
    import torch   # first: libglide_hip.so then binds to the HIP runtime torch has already loaded
    assert torch.cuda.is_available(), "bench.py needs an MI355X"
    from glide_amd import capi
    import bench_probes as probes
    capi.set_device(0)
    info = capi.device_info()

    if args.copy_calibration:
        import numpy as np
        nbytes = 1 << 30
        src, dst = capi.DeviceArray(nbytes // 4, np.uint32), capi.DeviceArray(nbytes // 4, np.uint32)
        probes.copy_bytes(dst, src, nbytes)
        e0, e1 = capi.Event(), capi.Event()
        e0.record()
        for _ in range(args.steps):
            probes.copy_bytes(dst, src, nbytes)
        e1.record()
        ms = e0.elapsed_ms(e1) / args.steps
        print(json.dumps({"kernel": "copy_kernel", "bytes_read": nbytes, "bytes_written": nbytes, "ms": ms,
                          "GBps_read_plus_write": 2 * nbytes / ms / 1e6}))
        return

    if args.valu_calibration:
        import numpy as np
        out = capi.DeviceArray(4, np.float32)
        rounds, res = 20000, {}
        for mode, (name, per_step) in enumerate((("fused multiply-add", 1), ("integer add", 1), ("compare + select", 2), ("DPP move + add", 2))):
            probes.valu_probe(mode, rounds, out)
            e0, e1 = capi.Event(), capi.Event()
            e0.record()
            for _ in range(args.steps):
                probes.valu_probe(mode, rounds, out)
            e1.record()
            ms = e0.elapsed_ms(e1) / args.steps
            insts = 2048 * 4 * rounds * 16 * per_step
            res[name] = {"wave_instructions": insts, "ms": ms, "G_wave_instructions_per_s": insts / ms / 1e6}
        print(json.dumps({"kernel": "valu_probe_kernel", "compute_units": info["compute_units"], "modes": res}))
        return

    if args.atomic_calibration:
        import numpy as np
        out = capi.DeviceArray(4, np.uint32)
        rounds, res = 256, {}
        ops = 2048 * 256 * rounds
        for name, slots in (("2 MB of slots (stays in L2)", 1 << 18), ("2 GB of slots (an offer table of 1M nodes)", 1 << 28)):
            for mode, kind in enumerate(("64-bit minimum, no result", "32-bit add, result used", "64-bit minimum, pairs of adjacent lanes on one 128-byte line",
                                         "64-bit minimum, 16 adjacent lanes on one 128-byte line")):
                table = capi.DeviceArray.full(2 * slots, 0xFFFFFFFF if mode == 0 else 0, np.uint32)
                probes.atomic_probe(mode, table, slots, rounds, out)
                e0, e1 = capi.Event(), capi.Event()
                e0.record()
                for _ in range(args.steps):
                    probes.atomic_probe(mode, table, slots, rounds, out)
                e1.record()
                ms = e0.elapsed_ms(e1) / args.steps
                res["%s; %s" % (kind, name)] = {"lane_operations": ops, "ms": ms, "G_lane_operations_per_s": ops / ms / 1e6}
                del table
        print(json.dumps({"kernel": "atomic_probe_kernel", "compute_units": info["compute_units"], "modes": res}))
        return

    if args.gather_calibration:
        import numpy as np
        out = capi.DeviceArray(4, np.float32)
        res = {}
        # (label, row bytes, row stride, rows per wave-wide step, table rows)
        for label, row_bytes, stride, rps, rows in (("128-byte rows (up to 128 dims as bytes), 8 lanes a row, 16 rows in flight per wavefront", 128, 128, 8, 1 << 20),
                                                    ("128-byte rows of a table of 4M, 8 lanes a row, 16 rows in flight per wavefront", 128, 128, 8, 1 << 22),
                                                    ("512-byte rows (128 dims), 8 lanes a row, 16 rows in flight per wavefront", 512, 512, 8, 1 << 20),
                                                    ("3840-byte rows (960 dims), 32 lanes a row, 8 rows in flight per wavefront", 3840, 3840, 2, 1 << 20),
                                                    ("3840-byte rows (960 dims), 64 lanes a row, 8 rows in flight per wavefront", 3840, 3840, 1, 1 << 20),
                                                    ("3840-byte rows 4096 bytes apart, 32 lanes a row, 8 rows in flight per wavefront", 3840, 4096, 2, 1 << 20),
                                                    ("3840-byte rows 3968 bytes apart, 32 lanes a row, 8 rows in flight per wavefront", 3840, 3968, 2, 1 << 20),
                                                    ("384-byte rows (96 dims), 8 lanes a row, 16 rows in flight per wavefront", 384, 384, 8, 1 << 20),
                                                    ("4096-byte rows (1024 dims), 32 lanes a row, 8 rows in flight per wavefront", 4096, 4096, 2, 1 << 20),
                                                    ("2048-byte rows (512 dims), 32 lanes a row, 8 rows in flight per wavefront", 2048, 2048, 2, 1 << 20)):
            table = capi.DeviceArray.full(rows * stride // 4, 0x3F800000, np.uint32)
            for waves_per_simd in (1, 2, 4, 8):
                waves = info["compute_units"] * 4 * waves_per_simd           # all resident at once: that many wavefronts per SIMD
                rows_per_wave = max(64, (4 << 30) // row_bytes // waves // 64 * 64)   # about 4 GiB per launch
                probes.gather_probe(table, rows, row_bytes, stride, waves, rows_per_wave, rps, out)
                e0, e1 = capi.Event(), capi.Event()
                e0.record()
                for _ in range(args.steps):
                    probes.gather_probe(table, rows, row_bytes, stride, waves, rows_per_wave, rps, out)
                e1.record()
                ms = e0.elapsed_ms(e1) / args.steps
                nbytes = waves * rows_per_wave * row_bytes
                res["%s; %d wavefronts" % (label, waves)] = {"bytes": nbytes, "ms": ms, "GBps": nbytes / ms / 1e6, "frac_of_8TBps": nbytes / ms / 1e6 / HBM_PEAK_GBS}
            del table
        print(json.dumps({"kernel": "gather_probe_kernel", "compute_units": info["compute_units"], "modes": res}))
        return

    if args.partition_only:
        import numpy as np
        from glide_amd import datasets as D
        num, dim, c = 1_000_000, 128, args.partition_only
        data = D.gmm_clipped(num, dim, seed=1234)
        d_data = capi.DeviceArray.from_numpy(data)
        d_cent = capi.DeviceArray.from_numpy(data[np.random.default_rng(7).permutation(num)[:c]].copy())
        d_idx, d_len = capi.DeviceArray((num, 3), np.uint32), capi.DeviceArray(c + 1, np.uint32)
        wb = capi.partition_assign_workspace_bytes(num, c)
        ws = capi.DeviceArray(wb // 4 + 1, np.uint32)
        run = lambda: capi.partition_assign(d_data, num, dim, d_cent, c, 1.04, 0, d_idx, d_len, None, ws, wb)
        for _ in range(args.warmup):
            run()
        e0, e1 = capi.Event(), capi.Event()
        e0.record()
        for _ in range(args.steps):
            run()
        e1.record()
        ms = e0.elapsed_ms(e1) / args.steps
        print(json.dumps({"stage": "partition assign (assign + scan + slot kernels)", "rows": num, "dim": dim, "centroids": c, "ms": ms,
                          "algorithmic_GBps": (num * dim * 4 + num * 12) / ms / 1e6, "algorithmic_TFLOPs": 2.0 * num * c * dim / ms / 1e9,
                          "fp32_mfma_peak_TFLOPs": 157.3}))
        return

    if args.knn_only:
        from glide_amd import index as G
        num, parts, knn_degree, nnd_iters, nq, desc, dim, metric, degree = WORKLOADS[args.workload]
        data, _ = make_data(args.workload, num, nq)
        d_data = capi.DeviceArray.from_numpy(data)
        res = {}
        pp = G.PartitionParameter(centroid_num=parts, boundary_factor=1.04, sample_factor=0.01, metric=metric)
        d_re, d_map, h_start, h_len, d_cent = G.preprocess(pp, d_data, res)
        nn = G.NNDescentParameter(graph_degree=knn_degree, max_iterations=args.nnd_iterations or nnd_iters)
        G.build_nnd(nn, d_re, h_start, h_len, res, stats=True)
        print(json.dumps({"stage": "NN-descent kNN graph", "workload": desc, "rows": int(h_len.sum()), "dim": dim, "k": knn_degree,
                          "iterations_allowed": nn.max_iterations, "knn_sec": res["knn_time"], "nnd_offers": res["nnd_stats"][0],
                          "nnd_offers_declined_by_threshold": res["nnd_stats"][1]}))
        return

    if args.workload == "cfg4":
        import bench_large
        print(json.dumps(bench_large.run(args, info), default=float))
        return

    main_res = run_workload(args, args.workload, torch, want_cpu=False if args.no_cpu else "full")
    details = {args.workload: main_res}
    emit_detail(args.workload, main_res)
    if args.workload == "cfg1" and not args.headline_only:
        for name in ("cfg1-navigable", "cfg0", "cfg2", "cfg3"):
            t0 = time.time()
            details[name] = run_workload(args, name, torch, want_cpu=not args.no_cpu)
            details[name]["wall_sec"] = time.time() - t0
            emit_detail(name, details[name])
    try:    # the whole record in one file, for whoever wants more than the stdout lines
        path = os.path.join(ROOT, args.details_file)
        os.makedirs(os.path.dirname(path), exist_ok=True)
        with open(path, "w") as f:
            json.dump(details, f, default=float, indent=1)
    except OSError:
        pass
    print(json.dumps(headline(args, args.workload, details, info["name"], args.details_file), default=float), flush=True)


DETAIL_KEYS = ("workload", "rows_read", "build_sec", "build_stages", "graph_recall_at_32", "graph_recall_at_32_global", "empty_slots_fraction", "beam",
               "recall_at_10", "recall_target_met", "reachable_recall_bound", "reachable_fraction_of_points", "qps", "ms_per_step", "kernel_ms",
               "nnd_iterations", "nnd_offers", "nnd_offers_declined_by_threshold", "sweep", "stage_rooflines", "roofline", "cpu_baseline", "wall_sec")


def emit_detail(name, res):
    """One stdout line per workload with everything measured on it; the compact headline line comes last."""
    print(json.dumps({"bench_detail": name, **{k: res[k] for k in DETAIL_KEYS if k in res}}, default=float), flush=True)


def headline(args, workload, details, device, details_file="the details file"):
    """The record's last stdout line: the fields of the benchmark contract for the headline workload, short enough (a few KB)
    that a consumer keeping only the tail of stdout still holds all of it.  `value` is the throughput of the timed steps;
    `metric` says what that is: the metric's operating point (the smallest beam with recall@10 >= 0.95) where the sweep
    reaches it, otherwise the widest named beam, with the bound the reference's entry rule puts on recall there."""
    r = details[workload]
    met = bool(r["recall_target_met"])
    r3 = lambda x: None if x is None else round(float(x), 4)
    if met:
        metric = "search QPS at recall@10 >= 0.95 (index build sec and graph recall@32 alongside), 1 MI355X"
    else:
        metric = ("search QPS at beam %d: recall@10 >= 0.95 is unreachable on this workload at any beam (reachable bound %.3f from the "
                  "reference's single entry point per partition); index build sec and graph recall@32 alongside, 1 MI355X"
                  % (r["beam"], r["reachable_recall_bound"]))
    roof = r["roofline"]
    line = {
        "metric": metric, "value": r["qps"], "unit": "queries/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": r["ms_per_step"], "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": r["workload"], "graph_degree": WORKLOADS[workload][8], "top_k": 10, "beam": r["beam"], "build_beam": 64,
                   "refine_beam": 128, "relaxant": 1.05, "boundary_factor": 1.04, "sample_factor": 0.01, "nnd_iterations": r["nnd_iterations"],
                   "nnd_termination_threshold": 1e-4},
        "rows_read": r.get("rows_read"), "device": device, "beam": r["beam"], "recall_at_10": r3(r["recall_at_10"]), "recall_target_met": met,
        "reachable_recall_bound": r3(r["reachable_recall_bound"]),
        "qps_at_recall_target": r["qps"] if met else None, "qps_at_max_beam": None if met else r["qps"],
        "build_sec": r3(r["build_sec"]), "build_stages": {k: r3(v) for k, v in r["build_stages"].items() if k != "detail"},
        "graph_recall_at_32": r3(r["graph_recall_at_32"]), "kernel_ms": r3(r["kernel_ms"]),
        "sweep": [dict(beam=x["beam"], recall_at_10=r3(x["recall_at_10"]), qps=round(x["qps"])) for x in r["sweep"]],
        "stage_fracs": {k: r3(v.get("frac")) for k, v in r["stage_rooflines"].items()},
        "roofline": {"bound": roof["bound"], "achieved": round(roof["achieved"], 1), "peak": roof["peak"], "unit": roof["unit"],
                     "frac": r3(roof["frac"]), "traffic": roof["traffic"], "kernel": roof["kernel"],
                     "algorithmic_bytes_per_launch": roof["algorithmic_bytes_per_launch"],
                     "scattered_row_ceiling_frac": r3(roof.get("scattered_row_ceiling_frac")),
                     "frac_of_scattered_row_ceiling": r3(roof.get("frac_of_scattered_row_ceiling"))},
    }
    if "cpu_baseline" in r:
        c = r["cpu_baseline"]
        line["cpu_baseline"] = {k: (r3(c[k]) if isinstance(c[k], float) else c[k])
                                for k in ("value", "unit", "cores", "kind", "sample", "recall_at_10", "nnd_points_per_sec", "bruteforce_qps") if k in c}
    # where the metric's operating point exists in this run: workload -> beam, QPS, recall, roofline fraction
    line["recall_target_met_on"] = {n: dict(beam=d["beam"], qps=round(d["qps"]), recall_at_10=r3(d["recall_at_10"]), roofline_frac=r3(d["roofline"]["frac"]),
                                            frac_of_scattered_row_ceiling=r3(d["roofline"].get("frac_of_scattered_row_ceiling")))
                                    for n, d in details.items() if d["recall_target_met"]}
    line["other_workloads"] = {n: dict(beam=d["beam"], qps=round(d["qps"]), recall_at_10=r3(d["recall_at_10"]), bound=r3(d["reachable_recall_bound"]),
                                       roofline_frac=r3(d["roofline"]["frac"]), build_sec=r3(d["build_sec"]))
                               for n, d in details.items() if n != workload}
    line["details"] = "one 'bench_detail' JSON line per workload earlier on stdout; " + details_file
    return line


if __name__ == "__main__":
    main()
