"""Host-side mirror of the reference's build/search interface on top of the C ABI.

Names, argument meaning and error behaviour follow the reference's C++ host layer:
  params.cuh           -> Metric, PartitionParameter, NNDescentParameter, IndexParameter, SearchParameter,
                          calculate_hash_bitlen, calculate_hash_reset_interval, adjust_search_params
  partition.cuh:159    -> preprocess()
  nn_descent.cuh:1405  -> build_nnd()
  glide.cuh:14-125     -> class GLIDE (ctor, load, build, search, accessors)
All device work goes through glide_amd.capi (libglide_hip.so); nothing here computes on the CPU beyond the
integer parameter arithmetic and the random choices the reference also makes on the host.
"""
import math
import time
from dataclasses import dataclass

import numpy as np

from . import capi

INVALID = 0xFFFFFFFF
BYTE_ROWS_DEGREE = 64      # the searches over rows of bytes take graphs of up to this degree
ROUGH_ROWS_DEGREE, ROUGH_ROWS_BEAM = 64, 128   # and the builds that look at rows in fp16 first this degree and beam


class Metric:
    Euclidean = capi.EUCLIDEAN
    Cosine = capi.COSINE


@dataclass
class PartitionParameter:          # params.cuh:10-15
    centroid_num: int = 10
    boundary_factor: float = 1.05
    sample_factor: float = 0.01
    metric: int = Metric.Euclidean
    kmeans_iterations: int = 20     # cuVS kmeans is replaced by greedy k-means++ seeding + Lloyd steps; count and seed are explicit here
    seed: int = 7


@dataclass
class NNDescentParameter:          # params.cuh:17-25
    graph_degree: int = 64
    intermediate_graph_degree: int = 0
    max_iterations: int = 20
    termination_threshold: float = 0.0001
    seed: int = 0

    def __post_init__(self):
        if not self.intermediate_graph_degree:
            self.intermediate_graph_degree = int(1.5 * self.graph_degree)


@dataclass
class IndexParameter:              # params.cuh:27-35
    graph_degree: int = 32
    knn_degree: int = 32
    relaxant_factor: float = 1.05
    metric: int = Metric.Euclidean
    seed: int = 11                  # the reference draws start points from std::random_device


@dataclass
class SearchParameter:             # params.cuh:37-47
    top_k: int = 10
    beam: int = 100
    max_iterations: int = 0
    min_iterations: int = 0
    hash_bit: int = 0
    hash_max_fill_rate: float = 0.5
    hashmap_min_bitlen: int = 0
    hash_reset_interval: int = 1
    search_block_size: int = 0


def calculate_hash_bitlen(beam, graph_degree, hashmap_max_fill_rate, hashmap_min_bitlen):   # params.cuh:49-66
    max_visited_nodes = beam + graph_degree
    min_bitlen, max_bitlen = 8, 13
    if min_bitlen < hashmap_min_bitlen:
        min_bitlen = hashmap_min_bitlen
    hash_bitlen = min_bitlen
    fill = np.float32(hashmap_max_fill_rate)
    while max_visited_nodes > np.float32(1 << hash_bitlen) * fill:
        hash_bitlen += 1
    return min(hash_bitlen, max_bitlen)


def calculate_hash_reset_interval(beam, graph_degree, hashmap_max_fill_rate, hash_bitlen):  # params.cuh:68-80
    interval = 1
    fill = np.float32(hashmap_max_fill_rate)
    while True:
        if beam + graph_degree * (interval + 1) > np.float32(1 << hash_bitlen) * fill:
            break
        interval += 1
    return interval


def adjust_search_params(min_iterations, max_iterations, beam):                            # params.cuh:82-99
    """Returns (max_iterations, beam)."""
    m = max_iterations
    if max_iterations == 0:
        m = int(1 + min(beam * 1.1, beam + 10.0))
    if max_iterations < min_iterations:
        m = min_iterations
    if max_iterations < m:
        max_iterations = m
    if beam % 32:
        beam += 32 - (beam % 32)
    return max_iterations, beam


def make_search_parameter(beam, degree, top_k=10):
    """SearchParameter sized the way the reference mains do (small_search.cu:102-108, small_build.cu:61-82)."""
    p = SearchParameter(top_k=top_k, beam=beam)
    p.max_iterations, p.beam = adjust_search_params(p.min_iterations, p.max_iterations, p.beam)
    p.hash_bit = calculate_hash_bitlen(p.beam, degree, p.hash_max_fill_rate, p.hashmap_min_bitlen)
    p.hash_reset_interval = calculate_hash_reset_interval(p.beam, degree, p.hash_max_fill_rate, p.hash_bit)
    return p


def _check_sizes(beam, degree):
    # kernel_config.cuh:48,60: std::invalid_argument("Unsupported beam" / "Unsupported graph_degree")
    if beam > 512 or (beam > 256 and beam % 16):     # the second: adjust_search_params rounds beams to multiples of 32
        raise ValueError("Unsupported beam")
    if degree > 256:
        raise ValueError("Unsupported graph_degree")


class _Timer:
    """GPU seconds between two events on the default stream (the reference sums cudaEvent intervals)."""

    def __init__(self):
        self.start, self.stop = capi.Event(), capi.Event()

    def __enter__(self):
        self.start.record()
        return self

    def __exit__(self, *exc):
        self.stop.record()
        self.seconds = self.start.elapsed_ms(self.stop) / 1000.0


def pad_rows(rows, multiple=4):
    """Points as the entry points want them: fp32 rows on the device whose length is a multiple of four values.  The
    reference's kernels loop over single values and take any dim (distance.cuh:9-27); here rows are read in 16-byte
    pieces, so points of another length get zeros behind them once, which changes no squared distance, inner product
    or norm.  numpy (num, dim) or DeviceArray in, DeviceArray (num, padded dim) out -- the same DeviceArray when its
    rows already fit, else a padded copy made on the device."""
    d = rows if isinstance(rows, capi.DeviceArray) else capi.DeviceArray.from_numpy(rows, np.float32)
    num, dim = d.shape
    held = (dim + multiple - 1) // multiple * multiple
    if held == dim:
        return d
    out = capi.DeviceArray((num, held), np.float32)
    capi.copy_rows(d, num, dim, out, held)
    capi.synchronize()
    if d is not rows:
        d.free()
    return out


def cut_rows(d_rows, dim):
    """The first `dim` values of every row of a DeviceArray of points, as numpy: centroids or reordered rows of padded
    points in the length the caller's data has."""
    num, held = d_rows.shape
    if held == dim:
        return d_rows.numpy()
    out = capi.DeviceArray((num, dim), np.float32)
    capi.copy_rows(d_rows, num, held, out, dim)
    capi.synchronize()
    h = out.numpy()
    out.free()
    return h


def try_array(nbytes):
    """nbytes on the device, or None where it has them not."""
    try:
        return capi.DeviceArray(nbytes, np.uint8)
    except capi.GlideHipError as e:
        if e.code != capi.OUT_OF_MEMORY:
            raise
        return None


def spare_array(nbytes):
    """Memory for a copy that only makes things faster, or None: what is free must have room for two of it, and none is made
    where the device has it in no one piece or another thread is faster."""
    return try_array(nbytes) if capi.mem_info()[0] // 2 >= nbytes else None


def byte_rows(d_rows):
    """The rows of a DeviceArray once more as bytes, for the searches over rows of whole numbers 0..255, as a DeviceArray;
    None where a value is none of those, rows of that length or so many are not held so, or memory is short."""
    num, dim = d_rows.shape
    nbytes = capi.byte_rows_bytes(num, dim)
    if nbytes == 0:
        return None
    d_other = capi.DeviceArray(1, np.uint32)
    for rows in (min(num, 2048), num):      # the first ones alone: rows of fractions end there
        d_bytes = spare_array(capi.byte_rows_bytes(rows, dim))
        if d_bytes is None:
            return None
        capi.pack_byte_rows(d_rows, rows, dim, d_bytes, d_other)
        if d_other.numpy()[0]:
            d_bytes.free()
            return None
        if rows == num:
            return d_bytes


def rough_rows_pay(num, dim):
    """Whether a build over `num` rows of `dim` values gains from a copy of them in fp16: the first look saves memory traffic and
    costs instructions and a second round of loads for the rows it leaves open.  Short rows leave lanes idle and gain later.
    Build with against without, in ms: 20 000 x 384 10.0 : 13.6, 20 000 x 200 7.5 : 7.8, 5 000 x 300 3.8 : 3.7; 120 000 x 128
    28.8 : 30.9, 70 000 x 128 17.4 : 17.2; 1 000 000 x 96 257 : 304, 234 567 x 96 56 : 53, 1 000 000 x 64 236 : 212.
    Sub-graphs to refinement alone: unit rows 200 000 x 112 34 : 46, 300 000 x 96 49 : 59, 600 000 x 96 100 : 138, 120 000 x 128 19 : 25;
    Beta-like rows, which share more of what they read, 200 000 x 112 42 : 43, 300 000 x 96 60 : 56, 700 000 x 96 145 : 156, 120 000 x 128
    23 : 22: the lines lie where neither loses."""
    return dim > 64 and 4 * num * dim >= (16 << 20 if dim >= 192 else 64 << 20 if dim >= 112 else 256 << 20)


def rough_rows(d_rows):
    """Rows once more in fp16, for the builds that look at them before they measure (half the memory traffic, the same results), as
    a DeviceArray; None where that does not pay, rows of that length are not looked at so, or memory is short."""
    num, dim = d_rows.shape
    nbytes = capi.rough_rows_bytes(num, dim) if rough_rows_pay(num, dim) else 0
    d_rough = spare_array(nbytes) if nbytes else None
    if d_rough is not None:
        capi.pack_rough_rows(d_rows, num, dim, d_rough)
    return d_rough


def rough_rows_help(d_rows, d_rough, d_graph, d_starts, d_lengths, d_start_points):
    """Whether the rows' distances are such that a look at them in fp16 tells most of those that need no measuring, and the searches
    such that the look saves traffic: from some rows and the graph that is there (see glide_hip_survey_rough_rows).
    Share told of the far ones, share of walks that arrive, and index with the copy against without, in ms: unit rows 250 000 x 128
    1.00, 1.0, 39 : 64; the same 16 standard deviations from the origin 0.97, 1.0, 41 : 64, 64 off 0.88, 39 : 45, 128 off 0.73,
    38 : 28.  60 000 x 960 at degree 64 0.97, 1.0, 158 : 258; 32 off 0.67, 180 : 210; 64 off 0.2, 221 : 219.  Dense clusters,
    60 000 x 384, 0.1, 0.1, 16.8 : 11.8.  Clusters far from each other, whose searches end in the wrong one, 200 000 x 128 0.99, 0.1,
    27 : 24, 60 000 x 384 0.98, 0.1, 18.7 : 18.9."""
    num, dim = d_rows.shape
    d_counts = capi.DeviceArray(4, np.uint32)
    capi.survey_rough_rows(d_rows, d_rough, num, dim, d_graph, d_graph.shape[1], d_starts, d_lengths, d_starts.shape[0], d_start_points, d_counts)
    far, told, rows, astray = (int(v) for v in d_counts.numpy())
    return far > 0 and told >= 0.6 * far and 2 * astray < rows


def _rows_read(d_bytes, d_rough):
    return "bytes" if d_bytes is not None else "fp16 first" if d_rough is not None else "fp32"


def draw_ids(num, count, seed, d_ids):
    """The first `count` entries of np.random.default_rng(seed).permutation(num) into a DeviceArray.  Returns the scratch of the
    device's draw (some 21 bytes a row; it may go once the draw is done), or None where the host has drawn: more rows than the
    device draws from, or no memory for it."""
    nbytes = capi.sample_ids_workspace_bytes(num)
    workspace = try_array(nbytes) if nbytes else None
    if workspace is None:
        d_ids.upload(np.random.default_rng(seed).permutation(num)[:count].astype(np.uint32))
    else:
        capi.sample_ids(num, count, seed, d_ids, workspace, nbytes)
    return workspace


def preprocess(param, d_data, result=None):
    """partition.cuh:159-193.  d_data: DeviceArray (num, dim) float32; rows of a length that is no multiple of four are
    padded (pad_rows), and the reordered rows and centroids returned then have the padded length (cut_rows gives them
    back in the data's own).

    Returns (d_reorder_data, d_map, h_segment_start, h_segment_length, d_centroids).  h_segment_* have
    centroid_num + 1 entries, the last being the boundary segment (start = num).
    """
    d_data = pad_rows(d_data)
    num, dim = d_data.shape
    c = param.centroid_num
    times = {}
    # get_centroids (partition.cuh:10-59): shuffle, sample, k-means on the sample
    sample_num = max(int(num * param.sample_factor), min(num, c))
    d_ids = capi.DeviceArray(sample_num, np.uint32)
    d_sample = capi.DeviceArray((sample_num, dim), np.float32)
    d_centroids = capi.DeviceArray((c, dim), np.float32)
    fit_bytes = capi.kmeans_workspace_bytes(c, dim)
    fit_ws = capi.DeviceArray(fit_bytes // 4 + 1, np.uint32)
    seed_bytes = capi.kmeans_seed_workspace_bytes(sample_num)
    seed_ws = capi.DeviceArray(seed_bytes // 8 + 1, np.uint64)
    ids_ws = draw_ids(num, sample_num, param.seed, d_ids)
    with _Timer() as t:
        capi.sample_rows(d_data, dim, d_ids, sample_num, d_sample)
        capi.kmeans_seed(d_sample, sample_num, dim, c, param.seed, d_centroids, seed_ws, seed_bytes)
        capi.kmeans_fit(d_sample, sample_num, dim, c, param.kmeans_iterations, d_centroids, fit_ws, fit_bytes)
    times["centroids"] = t.seconds
    for used in (ids_ws, d_ids, d_sample, seed_ws, fit_ws):     # before the reordered rows need their room
        if used is not None:
            used.free()
    # define_partition (partition.cuh:61-116)
    d_seg_idx = capi.DeviceArray((num, 3), np.uint32)
    d_seg_len = capi.DeviceArray(c + 1, np.uint32)
    wb = capi.partition_assign_workspace_bytes(num, c)
    ws = capi.DeviceArray(wb // 4 + 1, np.uint32)
    with _Timer() as t:
        capi.partition_assign(d_data, num, dim, d_centroids, c, param.boundary_factor, param.metric, d_seg_idx, d_seg_len,
                              None, ws, wb)
    times["assign"] = t.seconds
    h_len = d_seg_len.numpy()
    h_start = np.zeros(c + 1, dtype=np.uint32)
    h_start[1:] = np.cumsum(h_len[:-1], dtype=np.uint64).astype(np.uint32)
    reorder_num = num + int(h_len[c])
    # reorder (partition.cuh:118-157)
    d_reorder = capi.DeviceArray((reorder_num, dim), np.float32)
    d_map = capi.DeviceArray(reorder_num, np.uint32)
    d_start = capi.DeviceArray.from_numpy(h_start)
    with _Timer() as t:
        capi.reorder(d_data, num, dim, d_seg_idx, d_start, d_reorder, d_map)
    times["reorder"] = t.seconds
    if result is not None:
        result["pre_time"] = sum(times.values())
        result["pre_stages"] = times
    return d_reorder, d_map, h_start, h_len, d_centroids


def build_nnd(param, d_reorder_data, h_segment_start, h_segment_length, result=None, stats=False):
    """nn_descent.cuh:1405-1467.  Returns the kNN graph as a DeviceArray (reorder_num, graph_degree) of
    partition-local ids."""
    num, dim = d_reorder_data.shape
    degree = min(param.graph_degree, param.intermediate_graph_degree)
    d_ss = capi.DeviceArray.from_numpy(np.ascontiguousarray(h_segment_start, dtype=np.uint32))
    d_sl = capi.DeviceArray.from_numpy(np.ascontiguousarray(h_segment_length, dtype=np.uint32))
    d_knn = capi.DeviceArray((num, degree), np.uint32)
    wb = capi.nnd_workspace_bytes(num, dim, degree)
    ws = capi.DeviceArray(wb // 16 + 1, np.dtype("V16"))
    d_stats = capi.DeviceArray.from_numpy(np.zeros(2, np.uint64)) if stats else None
    with _Timer() as t:
        capi.nnd_build(d_reorder_data, num, dim, d_ss, d_sl, len(h_segment_start), degree, param.max_iterations,
                       param.termination_threshold, param.seed,
                       d_knn, ws, wb, d_stats)
    ws.free()
    if result is not None:
        result["knn_time"] = t.seconds
        if stats:
            result["nnd_stats"] = d_stats.numpy().tolist()
    return d_knn


class GLIDE:
    """glide.cuh:14-125 for Data_t = float, Index_t = uint32_t."""

    def __init__(self, graph_degree, data, centroids, metric):
        """data: numpy (num, dim) float32 or DeviceArray; centroids likewise (glide_impl.cuh:15-30).  Rows of a length
        that is no multiple of four are held padded (pad_rows); dim() is then the padded length."""
        _check_sizes(0, graph_degree)
        self.metric = metric
        self.d_data = pad_rows(data)
        self.d_centroids = pad_rows(centroids)
        if self.d_centroids.shape[1] != self.d_data.shape[1]:
            raise ValueError("centroids of %d values for points of %d" % (self.d_centroids.shape[1], self.d_data.shape[1]))
        self._graph_degree = int(graph_degree)
        self.d_graph = capi.DeviceArray((self.num(), self._graph_degree), np.uint32)
        self.d_start_points = None
        self._bytes = None      # (rows as bytes, the array they were made from, its write count)

    # accessors (glide.cuh:81-125)
    def dim(self): return self.d_data.shape[1]
    def num(self): return self.d_data.shape[0]
    def graph_degree(self): return self._graph_degree
    def centroid_num(self): return self.d_centroids.shape[0]
    def start_point_num(self): return self.d_start_points.shape[0]
    def data_view(self): return self.d_data
    def graph_view(self): return self.d_graph
    def centroid_view(self): return self.d_centroids
    def start_point_view(self): return self.d_start_points

    def _hold_byte_rows(self):
        """The index's rows as bytes, made anew (load, build): where they are whole numbers 0..255 its searches read a quarter
        of the memory and measure distances in integer arithmetic, with the same results to the bit."""
        self._bytes = None
        writes = self.d_data.writes
        d_bytes = byte_rows(self.d_data) if self._graph_degree <= BYTE_ROWS_DEGREE else None
        if d_bytes is not None:
            self._bytes = d_bytes, self.d_data, writes
        return d_bytes

    def _byte_rows(self):
        """The rows as bytes, or None: there are none, or the rows may have been written since.  A search then reads the rows,
        and so do all that follow: the copy goes."""
        held = self._bytes      # read once: another thread's search may let the copy go
        if held is None:
            return None
        d_bytes, made_from, writes = held
        if made_from is self.d_data and writes == made_from.writes and not made_from.shared:
            return d_bytes
        self._bytes = None
        return None

    def load(self, h_graph, h_start_points):                                   # glide_impl.cuh:32-41
        self.d_graph.upload(np.ascontiguousarray(h_graph, dtype=np.uint32))
        self.d_start_points = capi.DeviceArray.from_numpy(np.ascontiguousarray(h_start_points, dtype=np.uint32))
        self._bytes = None
        if not self.d_data.shared:
            self._hold_byte_rows()

    def start_point_select(self, h_segment_start, h_segment_length, h_map, seed):   # glide_impl.cuh:43-75
        rng = np.random.default_rng(seed)
        c = self.centroid_num()
        reorder_sp = np.zeros(len(h_segment_start), dtype=np.uint32)
        sp = np.zeros(c, dtype=np.uint32)
        for i in range(len(h_segment_start)):
            length = int(h_segment_length[i])
            reorder_sp[i] = rng.integers(0, length) if length > 0 else 0   # the reference underflows on an empty segment
            if i != c:
                sp[i] = h_map[int(h_segment_start[i]) + int(reorder_sp[i])] if length > 0 else 0
        return reorder_sp, sp

    def build(self, build_param, search_param_knn, search_param_refine, d_knn_graph, h_segment_start, h_segment_length,
              d_map, d_reorder_data, result=None, counters=False):
        """glide_impl.cuh:319-368: start points -> sub-graph build + boundary merge -> reverse edges -> refine.
        d_knn_graph, d_map and d_reorder_data are consumed (freed), as the reference resets its optionals."""
        num, dim, deg = self.num(), self.dim(), self._graph_degree
        knn_degree = d_knn_graph.shape[1]
        _check_sizes(search_param_knn.beam, knn_degree)
        _check_sizes(search_param_refine.beam, deg)
        reorder_num = d_reorder_data.shape[0]
        h_map = d_map.numpy()
        reorder_sp, sp = self.start_point_select(h_segment_start, h_segment_length, h_map, build_param.seed)
        d_ss = capi.DeviceArray.from_numpy(np.ascontiguousarray(h_segment_start, dtype=np.uint32))
        d_sl = capi.DeviceArray.from_numpy(np.ascontiguousarray(h_segment_length, dtype=np.uint32))
        d_rsp = capi.DeviceArray.from_numpy(reorder_sp)
        cnt = capi.new_counters() if counters else None
        times = {}
        p = search_param_knn
        with _Timer() as t:
            d_bytes = byte_rows(d_reorder_data) if knn_degree <= BYTE_ROWS_DEGREE else None
            d_rough = rough_rows(d_reorder_data) if d_bytes is None and knn_degree <= ROUGH_ROWS_DEGREE and p.beam <= ROUGH_ROWS_BEAM else None
            helps = None      # whether a look in fp16 helps; not known yet
            if d_rough is not None:
                helps = rough_rows_help(d_reorder_data, d_rough, d_knn_graph, d_ss, d_sl, d_rsp)
                if not helps:
                    d_rough.free()
                    d_rough = None
            rows_read = dict(subgraph=_rows_read(d_bytes, d_rough))
            capi.build_subgraph(d_reorder_data, num, dim, d_knn_graph, knn_degree, d_map, d_ss, d_sl, len(h_segment_start), d_rsp,
                                deg, p.beam, p.max_iterations, p.min_iterations, p.hash_bit, p.hash_reset_interval,
                                build_param.relaxant_factor, self.metric, self.d_graph, cnt, byte_rows=d_bytes, rough_rows=d_rough)
        times["subgraph"] = t.seconds
        with _Timer() as t:
            if reorder_num > num:
                capi.build_boundary(d_reorder_data, num, reorder_num, dim, d_knn_graph, knn_degree, d_map,
                                    int(reorder_sp[self.centroid_num()]), deg, p.beam, p.max_iterations, p.min_iterations,
                                    p.hash_bit, p.hash_reset_interval, build_param.relaxant_factor, self.metric, self.d_graph, cnt,
                                    byte_rows=d_bytes, rough_rows=d_rough)
        times["boundary"] = t.seconds
        if counters and result is not None:
            capi.synchronize()
            result["build_counters"] = capi.read_counters(cnt)
        capi.synchronize()
        for consumed in (d_knn_graph, d_reorder_data, d_bytes, d_rough):     # d_map is kept until the refine stage, which uses it as its order
            if consumed is not None:
                consumed.free()
        self.d_start_points = capi.DeviceArray.from_numpy(sp)
        # reverse_graph (glide_impl.cuh:194-256)
        d_rev = capi.DeviceArray((num, deg), np.uint32)
        d_rcnt = capi.DeviceArray(num, np.uint32)
        wb = capi.reverse_edges_workspace_bytes(num, deg)
        ws = capi.DeviceArray(wb // 8 + 1, np.uint64)
        with _Timer() as t:
            capi.reverse_edges(self.d_graph, num, deg, d_rev, d_rcnt, ws, wb)
            capi.insert_reverse(self.d_graph, d_rev, d_rcnt, num, deg)
        times["reverse"] = t.seconds
        ws.free()
        d_rcnt.free()
        # refine (glide_impl.cuh:258-316); d_rev is reused as the output graph
        times["refine"] = 0.0
        if search_param_refine.beam != 0:
            p = search_param_refine
            cnt2 = capi.new_counters() if counters else None
            with _Timer() as t:
                d_bytes = self._hold_byte_rows()
                may = d_bytes is None and helps is not False and deg <= ROUGH_ROWS_DEGREE and p.beam <= ROUGH_ROWS_BEAM
                d_rough = rough_rows(self.d_data) if may else None
                if d_rough is not None and helps is None and not rough_rows_help(self.d_data, d_rough, self.d_graph, *self._one_segment()):
                    d_rough.free()
                    d_rough = None
                rows_read["refine"] = _rows_read(d_bytes, d_rough)
                capi.refine(self.d_data, num, dim, self.d_graph, d_rev, deg, self.d_centroids, self.centroid_num(),
                            self.d_start_points, p.beam, p.max_iterations, p.min_iterations, p.hash_bit, p.hash_reset_interval,
                            build_param.relaxant_factor, self.metric, cnt2, order=d_map,
                            byte_rows=d_bytes, rough_rows=d_rough)
            times["refine"] = t.seconds
            del d_bytes
            self._byte_rows()      # the searches may not use them: rows whose address is known to others
            if d_rough is not None:
                d_rough.free()
            self.d_graph, d_rev = d_rev, self.d_graph
            if counters and result is not None:
                result["refine_counters"] = capi.read_counters(cnt2)
        elif not self.d_data.shared:
            self._hold_byte_rows()
        d_rev.free()
        d_map.free()
        if result is not None:
            result["rows_read"] = rows_read
            result["index_time"] = times["subgraph"] + times["boundary"] + times["reverse"]
            result["refine_time"] = times["refine"]
            result["build_stages"] = times

    def _one_segment(self):
        """Start, length and start point of all rows taken as one segment."""
        return (capi.DeviceArray.from_numpy(np.array([v], dtype=np.uint32)) for v in (0, self.num(), self.d_start_points.numpy()[0]))

    def search(self, param, d_query, result=None, counters=None, stream=None, out=None):
        """glide_impl.cuh:370-454.  d_query: DeviceArray (query_num, dim), in the data's own row length or padded as
        the data is held.  Returns (ids, dists) as numpy arrays unless `out` = (d_ids, d_dists) is given, in which case
        nothing is copied back."""
        _check_sizes(param.beam, self._graph_degree)
        d_query = pad_rows(d_query)
        if d_query.shape[1] != self.dim():
            raise ValueError("queries of %d values for points of %d" % (d_query.shape[1], self.dim()))
        nq = d_query.shape[0]
        if out is not None:
            d_ids, d_dists = out
        else:      # ids and distances in one allocation: one to make and free, and one copy back
            d_both = capi.DeviceArray((2, nq, param.top_k), np.uint32)
            d_ids, d_dists = d_both.ptr, d_both.ptr + d_both.nbytes // 2
        with _Timer() as t:
            capi.search(self.d_data, self.num(), self.dim(), self.d_graph, self._graph_degree, self.d_centroids, self.centroid_num(),
                        self.d_start_points, d_query, nq, param.top_k, param.beam, param.max_iterations, param.min_iterations,
                        param.hash_bit, param.hash_reset_interval, self.metric, d_ids, d_dists, counters, stream, byte_rows=self._byte_rows())
        if result is not None:
            result["search_time"] = t.seconds
            result["QPS"] = nq / t.seconds if t.seconds > 0 else float("inf")
        if out is not None:
            return None
        both = d_both.numpy()
        return both[0], both[1].view(np.float32)
