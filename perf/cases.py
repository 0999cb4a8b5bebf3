"""The work that programs built on this framework give it, as timed cases: index builds, partitioning and searches through
the Python host layer (glide_amd.index) and, for the per-partition search, the C ABI binding (glide_amd.capi).

`listed()` holds the cases by name, `draw(rng)` gives further ones of the same ranges; `prepare` makes what a program has
in hand before the call, `run` is one pass, `work` what a pass cannot do without and `tolerance` how far the outputs of
two correct implementations may be apart.

Points come in the distributions of glide_amd/datasets.py, drawn on the GPU from the seed:
  bytes     integers 0..255 of low intrinsic dimension, as image descriptors are (lowdim_integer)
  mixture   a clipped, rounded Gaussian mixture (gmm_clipped), the benchmark's medium configuration
  unit      unit-norm float rows for the cosine metric, a mixture on a low-dimensional cloud
  beta      Beta-like floats in [0, 1] scaled per cluster (beta_scaled), the 960-dim configuration
"""
import math

import numpy as np
import torch

from glide_amd import capi
from glide_amd import index as G


def listed():
    return [
        # One user's query against a million descriptors: the latency of a single search and everything around it.
        dict(name="search_one", kind="search", data="bytes", num=1_000_000, dim=128, parts=16, degree=32, queries=1, beam=32, top_k=10, host=True),
        # A small serving batch on long embedding rows (960 dims, degree 64), answers wanted on the host.
        dict(name="search_60_long_rows", kind="search", data="beta", num=60_000, dim=960, parts=8, degree=64, queries=60, beam=128, top_k=10, host=True),
        # The batch of the benchmark at its high-recall operating point: 10 000 queries, beam 64.
        dict(name="search_10k", kind="search", data="bytes", num=1_000_000, dim=128, parts=16, degree=32, queries=10_000, beam=64, top_k=10, host=False),
        # The benchmark's headline: 10 000 queries at beam 256 on the mixture.
        dict(name="search_10k_wide", kind="search", data="mixture", num=1_000_000, dim=128, parts=16, degree=32, queries=10_000, beam=256, top_k=10, host=False),
        # Cosine search for a re-ranking stage: 100 results for an odd number of float queries.
        dict(name="search_cosine_top100", kind="search", data="unit", num=300_000, dim=96, parts=12, degree=48, queries=2_347, beam=160, top_k=100, host=True),
        # The large path: every query searches the three or so partitions nearest to it, heads merged.
        dict(name="search_partitions", kind="partitions", data="bytes", num=500_000, dim=128, parts=64, degree=32, queries=5_000, beam=96, top_k=10),
        # Locality partitioning as the unmerged large path does it: 256 centroids, no boundary copies.
        dict(name="preprocess_256", kind="preprocess", data="bytes", num=2_000_000, dim=128, parts=256),
        # A small index built whole (a test set, a shard that is rebuilt often): launches and allocations count.
        dict(name="build_20k", kind="build", data="bytes", num=20_000, dim=100, parts=4, degree=32, knn_degree=32, rounds=20),
        # The small configuration of the benchmark: 100k x 128, kNN degree 64, eight rounds.
        dict(name="build_100k", kind="build", data="mixture", num=100_000, dim=128, parts=10, degree=32, knn_degree=64, rounds=8),
        # The cosine configuration, float rows, an odd size.
        dict(name="build_cosine", kind="build", data="unit", num=234_567, dim=96, parts=12, degree=32, knn_degree=32, rounds=20),
        # Long rows: 960 dims at degree 64.
        dict(name="build_long_rows", kind="build", data="beta", num=60_000, dim=960, parts=8, degree=64, knn_degree=64, rounds=20),
        # The benchmark's build: a million rows, degree 32, up to 20 rounds.
        dict(name="build_1m", kind="build", data="mixture", num=1_000_000, dim=128, parts=16, degree=32, knn_degree=32, rounds=20),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case.  Row lengths are those of common embeddings and descriptors, odd ones among them; sizes are limited
    so that no drawn case costs more than the largest listed one."""
    kind = rng.choice(["search", "search", "search", "build", "build", "preprocess", "partitions"])
    data = rng.choice(["bytes", "bytes", "mixture", "unit", "beta"])
    dim = rng.choice([25, 50, 64, 96, 100, 128, 128, 160, 200, 256, 300, 384, 512, 768, 960, rng.randint(20, 1000)])
    longer = max(1.0, dim / 128.0)
    if kind == "search":
        degree = rng.choice([16, 24, 32, 32, 32, 40, 48, 56, 64, 96])
        num = _log(rng, 20_000, min(1_000_000, 900_000 / (longer * max(1.0, degree / 32.0) ** 2)))
        beam = rng.choice([32, 32, 64, 64, 96, 128, 160, 192, 256, 320, 512])
        top_k = rng.choice([1, 10, 10, 10, min(beam, rng.randint(11, 100))])
        queries = _log(rng, 1, 10_000)
        return dict(kind=kind, data=data, num=num, dim=dim, parts=rng.randint(2, 24), degree=degree, queries=queries, beam=beam, top_k=top_k,
                    host=rng.random() < 0.5)
    if kind == "build":
        degree = rng.choice([24, 32, 32, 48, 64])
        knn_degree = max(degree, rng.choice([32, 32, 64]))
        num = _log(rng, 5_000, 500_000 / (longer * max(1.0, knn_degree / 32.0) ** 2))
        return dict(kind=kind, data=data, num=num, dim=dim, parts=rng.randint(2, 16), degree=degree, knn_degree=knn_degree, rounds=rng.choice([8, 12, 20]))
    if kind == "preprocess":
        parts = _log(rng, 4, 256)
        return dict(kind=kind, data=data, num=_log(rng, 50_000, 2_000_000 / longer), dim=dim, parts=parts)
    return dict(kind=kind, data=data, num=_log(rng, 50_000, 400_000 / longer), dim=dim, parts=rng.randint(8, 48), degree=rng.choice([16, 32, 32]),
                queries=_log(rng, 100, 5_000), beam=rng.choice([32, 64, 96, 128]), top_k=rng.choice([1, 10, 10, 30]))


# ---------------------------------------------------------------------------------------------------------- inputs
def _points(data, num, dim, which, seed):
    """fp32 rows on the GPU.  `which` separates the rows of the index (0) from the queries (1); both come from one
    distribution, which the seed fixes."""
    shape = torch.Generator(device="cuda").manual_seed(1_000_003 * seed + 17)
    r = torch.Generator(device="cuda").manual_seed(1_000_003 * seed + 1_001 + which)
    normal = lambda *s, g=r: torch.randn(*s, generator=g, device="cuda")              # noqa: E731
    if data == "bytes":
        a = normal(12, dim, g=shape)
        x = normal(num, 12) @ a * 20.0 + 128.0 + normal(num, dim) * 3.0
        return x.clamp_(0.0, 255.0).round_()
    if data == "mixture":
        means = torch.rand(64, dim, generator=shape, device="cuda") * 160.0
        x = means[torch.randint(0, 64, (num,), generator=r, device="cuda")] + normal(num, dim) * 25.0
        return x.clamp_(0.0, 255.0).round_()
    if data == "unit":
        a = normal(10, dim, g=shape)
        means = normal(64, 10, g=shape)
        x = (means[torch.randint(0, 64, (num,), generator=r, device="cuda")] + normal(num, 10)) @ a + normal(num, dim) * 0.1
        return x / x.norm(dim=1, keepdim=True)
    scales = torch.rand(128, dim, generator=shape, device="cuda") * 0.95 + 0.05
    x = torch.rand(num, dim, generator=r, device="cuda")
    return (1.0 - x.sqrt()).square_() * scales[torch.randint(0, 128, (num,), generator=r, device="cuda")]


def _device_array(rows):
    """The framework's own device array with a copy of a tensor's rows."""
    out = capi.DeviceArray(tuple(rows.shape), np.float32)
    capi.copy_rows(rows.contiguous(), rows.shape[0], rows.shape[1], out, rows.shape[1])
    capi.synchronize()
    return out


class _Memory:
    """A device array as other libraries read it; keeps the array alive."""

    def __init__(self, array):
        self.array = array
        kind = "<f4" if array.dtype == np.float32 else "<i4"
        self.__cuda_array_interface__ = dict(shape=array.shape, typestr=kind, data=(array.ptr, False), strides=None, version=2)


def _tensor(array):
    return torch.as_tensor(_Memory(array), device="cuda")


def _metric(case):
    return G.Metric.Cosine if case["data"] == "unit" else G.Metric.Euclidean


def _build(points, case):
    """A finished index over `points` as the benchmark and test.sh build it: build beam 64, refine beam 128."""
    param = G.PartitionParameter(centroid_num=case["parts"], boundary_factor=1.04, sample_factor=0.01, metric=_metric(case))
    d_reorder, d_map, starts, lengths, d_centroids = G.preprocess(param, points)
    knn_degree = case.get("knn_degree", case["degree"])
    d_knn = G.build_nnd(G.NNDescentParameter(graph_degree=knn_degree, max_iterations=case.get("rounds", 20)), d_reorder, starts, lengths)
    index = G.GLIDE(case["degree"], points, d_centroids, _metric(case))
    index.build(G.IndexParameter(graph_degree=case["degree"], knn_degree=knn_degree, relaxant_factor=1.05, metric=_metric(case)),
                G.make_search_parameter(64, knn_degree), G.make_search_parameter(128, knn_degree), d_knn, starts, lengths, d_map, d_reorder)
    return index, starts, lengths


def _build_partitions(points, case):
    """Sub-graphs of every partition by themselves, resident on the GPU, as the large path keeps them: no boundary copies;
    sub-graph build, reverse edges and refine per partition."""
    param = G.PartitionParameter(centroid_num=case["parts"], boundary_factor=0.0, sample_factor=0.01, metric=_metric(case))
    d_rows, d_map, starts, lengths, d_centroids = G.preprocess(param, points)
    c, degree = case["parts"], case["degree"]
    starts, lengths = starts[:c], lengths[:c]
    num, dim = d_rows.shape
    d_knn = G.build_nnd(G.NNDescentParameter(graph_degree=degree), d_rows, starts, lengths)
    d_built, d_graph = capi.DeviceArray((num, degree), np.uint32), capi.DeviceArray((num, degree), np.uint32)
    most = int(lengths.max())
    d_reverse, d_counts = capi.DeviceArray((most, degree), np.uint32), capi.DeviceArray(most, np.uint32)
    bytes_ = capi.reverse_edges_workspace_bytes(most, degree)
    workspace = capi.DeviceArray(bytes_ // 8 + 1, np.uint64)
    b, r = G.make_search_parameter(64, degree), G.make_search_parameter(128, degree)
    entries = np.full(c, capi.INVALID, np.uint32)
    for s in range(c):
        first, n = int(starts[s]), int(lengths[s])
        if n == 0:
            continue
        entries[s] = n // 2
        rows, built = d_rows.ptr + 4 * dim * first, d_built.ptr + 4 * degree * first
        capi.build_segment(rows, n, dim, d_knn.ptr + 4 * degree * first, degree, n // 2, degree, b.beam, b.max_iterations, b.min_iterations, b.hash_bit,
                           b.hash_reset_interval, 1.05, _metric(case), built)
        capi.reverse_edges(built, n, degree, d_reverse, d_counts, workspace, bytes_)
        capi.insert_reverse(built, d_reverse, d_counts, n, degree)
        capi.refine_segment(rows, n, dim, built, d_graph.ptr + 4 * degree * first, degree, n // 2, r.beam, r.max_iterations, r.min_iterations, r.hash_bit,
                            r.hash_reset_interval, 1.05, _metric(case))
    capi.synchronize()
    return dict(rows=d_rows, graph=d_graph, map=d_map, starts=capi.DeviceArray.from_numpy(np.ascontiguousarray(starts)),
                entries=capi.DeviceArray.from_numpy(entries), centroids=d_centroids)


def prepare(case, seed):
    state = dict(case=case)
    points = _device_array(_points(case["data"], case["num"], case["dim"], 0, seed))
    if case["kind"] in ("build", "preprocess"):
        state["points"] = points
        return state
    queries = _points(case["data"], case["queries"], case["dim"], 1, seed)
    shape = (case["queries"], case["top_k"])
    if case["kind"] == "search":
        state["index"] = _build(points, case)[0]
        state["param"] = G.make_search_parameter(case["beam"], case["degree"], case["top_k"])
        state["queries"] = _device_array(queries)
        if not case["host"]:       # a serving loop keeps its result buffers
            state["out"] = (torch.empty(shape, dtype=torch.int32, device="cuda"), torch.empty(shape, dtype=torch.float32, device="cuda"))
        return state
    state["index"] = _build_partitions(points, case)
    state["param"] = G.make_search_parameter(case["beam"], case["degree"], case["top_k"])
    state["queries"] = G.pad_rows(_device_array(queries))
    state["segments"] = capi.DeviceArray((case["queries"], case["parts"]), np.uint32)
    state["out"] = (torch.empty(shape, dtype=torch.int32, device="cuda"), torch.empty(shape, dtype=torch.float32, device="cuda"))
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "search":
        if case["host"]:
            return state["index"].search(state["param"], state["queries"])
        state["index"].search(state["param"], state["queries"], out=state["out"])
        return state["out"]
    if case["kind"] == "partitions":
        x, p, q = state["index"], state["param"], state["queries"]
        dim = q.shape[1]
        capi.select_segments(q, case["queries"], dim, x["centroids"], case["parts"], 2, 1.1, _metric(case), state["segments"])
        capi.search_partitions(x["rows"], dim, x["graph"], case["degree"], x["map"], x["starts"], x["entries"], case["parts"], q, case["queries"],
                               state["segments"], case["top_k"], p.beam, p.max_iterations, p.min_iterations, p.hash_bit, p.hash_reset_interval,
                               _metric(case), *state["out"])
        return state["out"]
    if case["kind"] == "preprocess":
        param = G.PartitionParameter(centroid_num=case["parts"], boundary_factor=0.0, sample_factor=0.01, metric=_metric(case))
        d_reorder, d_map, starts, lengths, d_centroids = G.preprocess(param, state["points"])
        return _tensor(d_reorder), _tensor(d_map), starts, lengths, _tensor(d_centroids)
    index, starts, lengths = _build(state["points"], case)
    return _tensor(index.graph_view()), _tensor(index.start_point_view()), _tensor(index.centroid_view()), starts, lengths


def _searches(num, dim, degree, beam):
    """Bytes and operations of `num` beam searches that reach their rows one expansion after another: about one expansion
    a beam entry, each reading a graph row and, on average, the rows of the half of its neighbours not met before.  No two
    searches read the same rows, so every search pays for its own."""
    expansions = beam + 4
    rows = expansions * degree / 2
    return num * (expansions * degree * 4 + (rows + 1) * dim * 4), num * rows * dim * 3


def work(case):
    num, dim = case["num"], case["dim"]
    if case["kind"] in ("search", "partitions"):
        each = 3 if case["kind"] == "partitions" else 1          # two partitions a query at least, three on average
        b, f = _searches(case["queries"] * each, dim, case["degree"], case["beam"])
        return dict(bytes=b + case["queries"] * case["top_k"] * 8, flops=f)
    # partitioning: rows read for the assignment and again for the reordered copy, which is written
    partition = dict(bytes=3 * num * dim * 4 + num * 24, flops=2 * num * dim * case["parts"])
    if case["kind"] == "preprocess":
        return partition
    # NN-descent, a dozen rounds until it settles: 96 half-precision rows a list and round against 32 x (32 + 64) pairs
    rounds = min(case["rounds"], 12)
    join = dict(bytes=rounds * num * 96 * dim * 2, flops=rounds * num * 32 * 96 * dim * 2)
    b1, f1 = _searches(num, dim, case["knn_degree"], 64)
    b2, f2 = _searches(num, dim, case["degree"], 128)
    return dict(bytes=partition["bytes"] + join["bytes"] + b1 + b2 + num * case["degree"] * 4, flops=partition["flops"] + join["flops"] + f1 + f2)


def tolerance(case):
    """Four times what the outputs move by when every sum over a row is taken in another order (the dims of rows, centroids
    and queries permuted).  Searches: distances by 6e-8 (3e-7 of one value at most) and no id, but ids may change places
    where two distances agree to that precision.  Builds on integer rows: nothing, their sums are exact.  Builds on float
    rows carry a change on -- a point that goes to another partition, or a list that orders two candidates the other way,
    changes the rows of the graph around it: 1e-4 of the ids on 96-dim unit rows, a quarter of them on 960-dim rows, where
    the most that can still be called the same result is stated instead.  Partitioning: a point that changes its partition
    moves all that follow it."""
    if case["kind"] in ("search", "partitions"):
        return dict(rel=3e-7, max=2e-6, differ=1e-3)
    if case["kind"] == "build" and case["data"] in ("bytes", "mixture"):
        return dict(rel=1e-6, max=1e-5, differ=1e-4)
    if case["kind"] == "build" and case["dim"] <= 128:
        return dict(rel=1e-6, max=1e-5, differ=5e-4)
    return dict(rel=1e-6, max=1e-5, differ=0.01)
