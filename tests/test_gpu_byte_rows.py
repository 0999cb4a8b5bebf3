"""Searches, sub-graph builds and refinement over rows held as bytes against the same calls on the fp32 rows: sums of squares
of up to 256 whole numbers 0..255 are exact in fp32 and in integers, so ids, distances, graphs and counters must agree to the
bit.  Rows and queries reach both ends of the range (256 dims of 0 against 255 give the largest sum there is)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INV = 0xFFFFFFFF


@pytest.fixture(scope="module")
def hip():
    from glide_amd import capi
    capi.set_device(0)
    return capi


def rows_of(rng, n, dim):
    """Clustered bytes, a fifth of the values at the ends of the range, some rows equal, one all 0 and one all 255."""
    x = rng.integers(0, 256, (8, dim))[rng.integers(0, 8, n)] + rng.integers(-20, 21, (n, dim))
    x = np.clip(x, 0, 255)
    x[rng.random((n, dim)) < 0.1] = 0
    x[rng.random((n, dim)) < 0.1] = 255
    x[n // 2: n // 2 + 5] = x[3]
    x[0], x[1] = 0, 255
    return x.astype(np.float32)


def packed(hip, rows):
    d = hip.DeviceArray.from_numpy(rows)
    n, dim = rows.shape
    d_bytes, d_other = hip.DeviceArray.full(hip.byte_rows_bytes(n, dim) // 4, 0xDEADBEEF), hip.DeviceArray.full(1, 7)
    hip.pack_byte_rows(d, n, dim, d_bytes, d_other)
    return d, d_bytes, int(d_other.numpy()[0])


@pytest.mark.parametrize("n,dim", [(1, 4), (33, 100), (700, 128), (2049, 132), (5000, 256)])
def test_packed_rows(hip, n, dim):
    rows = rows_of(np.random.default_rng(n), max(n, 8), dim)[:n]
    _, d_bytes, other = packed(hip, rows)
    held = d_bytes.numpy().view(np.uint8).reshape(n, 128 if dim <= 128 else 256)
    assert other == 0 and np.array_equal(held[:, :dim], rows) and not held[:, dim:].any()
    for value, at in ((0.5, (n - 1, dim - 1)), (-1.0, (n // 2, 0)), (256.0, (0, dim // 2)), (np.nan, (n - 1, 3)), (np.inf, (0, 0)), (254.99998, (n // 3, 1))):
        bad = rows.copy()
        bad[at] = value
        assert packed(hip, bad)[2] == 1, (value, at)
    rows[n - 1, 0] = -0.0      # the same number as 0
    assert packed(hip, rows)[2] == 0


def test_lengths_that_are_not_held(hip):
    assert hip.byte_rows_bytes(100, 260) == 0 and hip.byte_rows_bytes(100, 6) == 0 and hip.byte_rows_bytes(100, 256) == 25600
    d = hip.DeviceArray((4, 260), np.float32)
    with pytest.raises(hip.GlideHipError):
        hip.pack_byte_rows(d, 4, 260, hip.DeviceArray(4096, np.uint8), hip.DeviceArray(1, np.uint32))


CASES = [(dim, degree, beam, metric) for i, (dim, degree) in enumerate([(4, 8), (16, 32), (100, 24), (128, 32), (128, 64), (132, 40), (200, 64), (256, 32)])
         for beam, metric in [((32, 64, 128, 256)[i % 4], i % 2), ((512, 288, 160, 96)[i % 4], 1 - i % 2)]]


@pytest.mark.parametrize("dim,degree,beam,metric", CASES)
def test_search(hip, dim, degree, beam, metric):
    from oracle import oracle as O
    rng = np.random.default_rng(dim + degree + beam)
    n, nq, c = 900, 70, 3
    rows = rows_of(rng, n, dim)
    knn, _ = O.bruteforce_knn(rows, rows, degree, exclude_self=True)
    knn[rng.random(knn.shape) < 0.05] = INV
    queries = rows_of(rng, nq, dim)
    queries[2] = rows[7]
    odd = {5: 0.25, 11: -3.0, 30: 300.0, 41: 127.00001, nq - 1: 1e-30}       # queries that are not of bytes
    for q, v in odd.items():
        queries[q, dim - 1] = v
    queries[50, 0] = np.nan
    queries[51, 0] = -0.0
    d, d_bytes, other = packed(hip, rows)
    assert other == 0
    sp = O.search_params(beam, degree)
    d_g, d_q = hip.DeviceArray.from_numpy(knn), hip.DeviceArray.from_numpy(queries)
    d_c, d_sp = hip.DeviceArray.from_numpy(rows[[10, 400, 800]] + 0.5), hip.DeviceArray.from_numpy(np.array([1, 0, 77], np.uint32))
    got = []
    for b in (None, d_bytes):
        ids, dists, cnt = hip.DeviceArray.full((nq, 10), 0xDEADBEEF), hip.DeviceArray.full((nq, 10), 0xDEADBEEF), hip.new_counters()
        hip.search(d, n, dim, d_g, degree, d_c, c, d_sp, d_q, nq, 10, sp["beam"], sp["max_iterations"], sp["min_iterations"], sp["hash_bit"],
                   sp["hash_reset_interval"], metric, ids, dists, cnt, byte_rows=b)
        hip.synchronize()
        got.append((ids.numpy(), dists.numpy(), hip.read_counters(cnt)))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]


@pytest.mark.parametrize("dim,knn_degree,degree,build_beam,refine_beam,metric",
                         [(4, 16, 8, 32, 64, 0), (100, 32, 32, 64, 128, 0), (128, 64, 32, 128, 256, 1), (128, 32, 64, 256, 512, 0), (132, 24, 40, 64, 128, 1),
                          (256, 64, 64, 320, 288, 0), (256, 32, 24, 64, 64, 1)])
def test_build_and_refine(hip, dim, knn_degree, degree, build_beam, refine_beam, metric):
    from oracle import oracle as O
    rng = np.random.default_rng(dim + degree)
    lengths, boundary = (400, 300), 120
    n = sum(lengths)
    rows = rows_of(rng, n, dim)
    reorder = np.concatenate([rows, rows[rng.permutation(n)[:boundary]]])
    mp = np.concatenate([rng.permutation(n), rng.permutation(n)[:boundary]]).astype(np.uint32)
    starts, lens = np.array([0, lengths[0], n], np.uint32), np.array([*lengths, boundary], np.uint32)
    knn = np.concatenate([O.bruteforce_knn(reorder[s:s + m], reorder[s:s + m], knn_degree, metric, exclude_self=True)[0] for s, m in zip(starts, lens)])
    knn[rng.random(knn.shape) < 0.05] = INV
    b, r = O.search_params(build_beam, knn_degree), O.search_params(refine_beam, max(knn_degree, degree))
    d_re, d_re_bytes, other = packed(hip, reorder)
    d_rows, d_rows_bytes, other2 = packed(hip, rows)
    assert other == 0 and other2 == 0
    up = hip.DeviceArray.from_numpy
    d_knn, d_map, d_s, d_l = up(knn), up(mp), up(starts), up(lens)
    d_sp, d_c, d_gsp = up(np.array([5, 9, 2], np.uint32)), up(rows[[20, 600]] + 0.25), up(np.array([3, 500], np.uint32))
    got = []
    for re_bytes, row_bytes in ((None, None), (d_re_bytes, d_rows_bytes)):
        g, out, cnt = hip.DeviceArray.full((n, degree), INV), hip.DeviceArray.full((n, degree), 0xDEADBEEF), hip.new_counters()
        args = (b["beam"], b["max_iterations"], b["min_iterations"], b["hash_bit"], b["hash_reset_interval"], 1.05, metric, g, cnt)
        hip.build_subgraph(d_re, n, dim, d_knn, knn_degree, d_map, d_s, d_l, 3, d_sp, degree, *args, byte_rows=re_bytes)
        hip.build_boundary(d_re, n, n + boundary, dim, d_knn, knn_degree, d_map, 2, degree, *args, byte_rows=re_bytes)
        hip.refine(d_rows, n, dim, g, out, degree, d_c, 2, d_gsp, r["beam"], r["max_iterations"], r["min_iterations"], r["hash_bit"],
                   r["hash_reset_interval"], 1.05, metric, cnt, order=d_map, byte_rows=row_bytes)
        hip.synchronize()
        got.append((g.numpy(), out.numpy(), hip.read_counters(cnt)))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]
    assert (got[0][1] != INV).any()


def test_index_follows_its_rows(hip):
    """Rows written after load() are the rows that are searched, whoever writes them."""
    from glide_amd import index as G
    from oracle import oracle as O
    rng = np.random.default_rng(3)
    n, dim, degree = 600, 64, 16
    first, second = rows_of(rng, n, dim), rows_of(rng, n, dim)
    knn, _ = O.bruteforce_knn(first, first, degree, exclude_self=True)
    sp, queries = G.make_search_parameter(64, degree), hip.DeviceArray.from_numpy(rows_of(rng, 20, dim))
    d = hip.DeviceArray.from_numpy(first)
    index = G.GLIDE(degree, d, first[:2], G.Metric.Euclidean)

    def fresh(rows):
        other = G.GLIDE(degree, rows + 0.0, first[:2], G.Metric.Euclidean)
        other.load(knn, np.array([4, 9], np.uint32))
        other._bytes = None
        return other.search(sp, queries)

    def agree(rows):
        return all(np.array_equal(a, b) for a, b in zip(index.search(sp, queries), fresh(rows)))

    index.load(knn, np.array([4, 9], np.uint32))
    assert index._byte_rows() is not None and agree(first)
    d.upload(second)
    assert index._byte_rows() is None and agree(second)
    index.load(knn, np.array([4, 9], np.uint32))
    assert index._byte_rows() is not None and agree(second)
    hip.copy_rows(hip.DeviceArray.from_numpy(first), n, dim, d, dim)
    assert index._byte_rows() is None and agree(first)
    index.load(knn, np.array([4, 9], np.uint32))
    assert index._byte_rows() is not None and agree(first)
    hip.copy_rows(hip.DeviceArray.from_numpy(second), n, dim, d.ptr, dim)     # by address: not seen as a write to `d`
    assert index._byte_rows() is None and agree(second)
    fractions = G.GLIDE(degree, first + 0.5, first[:2], G.Metric.Euclidean)
    fractions.load(knn, np.array([4, 9], np.uint32))
    assert fractions._byte_rows() is None


@pytest.mark.parametrize("dim,degree,beam,top_k,bad_row", [(100, 16, 64, 10, None), (128, 32, 96, 30, None), (128, 32, 64, 10, 2500), (128, 32, 64, 10, 5),
                                                            (256, 64, 256, 64, None), (132, 24, 512, 128, None)])
def test_partitions(hip, dim, degree, beam, top_k, bad_row):
    """Rows of a known number (a DeviceArray) are searched as bytes, the same rows by address as fp32."""
    from oracle import oracle as O
    rng = np.random.default_rng(dim + beam)
    lengths = (1500, 0, 1300, 200)
    n, c, nq = sum(lengths), len(lengths), 120
    rows = rows_of(rng, n, dim)
    if bad_row is not None:
        rows[bad_row, 1] += 0.5
    starts = np.concatenate([[0], np.cumsum(lengths)[:-1]]).astype(np.uint32)
    graph = np.concatenate([O.bruteforce_knn(rows[s:s + m], rows[s:s + m], degree, exclude_self=True)[0] for s, m in zip(starts, lengths) if m])
    entries = np.array([7, INV, 100, 0], np.uint32)
    queries = rows_of(rng, nq, dim)
    queries[3, 2], queries[nq - 1, 0], queries[40, 1] = 0.5, -1.0, np.nan
    segments = np.full((nq, c), INV, np.uint32)
    for q in range(nq):
        pick = rng.permutation(c)[:rng.integers(1, c + 1)]
        segments[q, :len(pick)] = pick
    sp = O.search_params(beam, degree)
    assert nq * beam * degree // 2 >= 4 * n
    up = hip.DeviceArray.from_numpy
    d, d_g, d_m, d_s, d_e, d_q, d_seg = up(rows), up(graph), up(rng.permutation(n).astype(np.uint32)), up(starts), up(entries), up(queries), up(segments)
    got = []
    for data in (d.ptr, d):
        ids, dists, cnt = hip.DeviceArray.full((nq, top_k), 0xDEADBEEF), hip.DeviceArray.full((nq, top_k), 0xDEADBEEF), hip.new_counters()
        hip.search_partitions(data, dim, d_g, degree, d_m, d_s, d_e, c, d_q, nq, d_seg, top_k, sp["beam"], sp["max_iterations"], sp["min_iterations"],
                              sp["hash_bit"], sp["hash_reset_interval"], 0, ids, dists, cnt)
        got.append((ids.numpy(), dists.numpy(), hip.read_counters(cnt)))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]
    assert (got[0][0][:, 0] < n).sum() >= nq // 2          # some select the empty partition alone


@pytest.mark.parametrize("refine_beam", [0, 128])
def test_bytes_that_no_search_may_use_are_not_kept(hip, refine_beam):
    """Once the address of the rows has been handed out an index searches its fp32 rows: it then holds no copy of them."""
    from glide_amd import index as G
    rng = np.random.default_rng(5)
    n, dim, degree = 3000, 64, 32
    rows = rows_of(rng, n, dim)
    sp, queries = G.make_search_parameter(64, degree), hip.DeviceArray.from_numpy(rows_of(rng, 50, dim))

    def build(d):
        d_reorder, d_map, starts, lengths, d_c = G.preprocess(G.PartitionParameter(centroid_num=3, boundary_factor=1.04, sample_factor=0.5), d)
        d_knn = G.build_nnd(G.NNDescentParameter(graph_degree=degree, max_iterations=6), d_reorder, starts, lengths)
        index = G.GLIDE(degree, d, d_c, G.Metric.Euclidean)
        index.build(G.IndexParameter(graph_degree=degree, knn_degree=degree, relaxant_factor=1.05), G.make_search_parameter(64, degree),
                    G.make_search_parameter(refine_beam, degree) if refine_beam else G.SearchParameter(beam=0), d_knn, starts, lengths, d_map, d_reorder)
        return index

    own, known = build(hip.DeviceArray.from_numpy(rows)), hip.DeviceArray.from_numpy(rows)
    assert known.ptr
    other = build(known)
    assert own._bytes is not None and other._bytes is None
    assert np.array_equal(own.d_graph.numpy(), other.d_graph.numpy())
    expect = own.search(sp, queries)
    assert all(np.array_equal(a, b) for a, b in zip(expect, other.search(sp, queries)))
    other.load(own.d_graph.numpy(), own.d_start_points.numpy())
    assert other._bytes is None and all(np.array_equal(a, b) for a, b in zip(expect, other.search(sp, queries)))
    assert own.d_data.ptr and own._bytes is not None       # handed out later: gone with the next search
    assert all(np.array_equal(a, b) for a, b in zip(expect, own.search(sp, queries))) and own._bytes is None


def test_partitions_without_room_for_the_bytes(hip, monkeypatch):
    """Rows as bytes are a copy in the workspace: where there is no memory for it the search takes the rows as they are."""
    from oracle import oracle as O
    rng = np.random.default_rng(9)
    n, dim, degree, nq, top_k = 4000, 64, 32, 200, 10
    rows = rows_of(rng, n, dim)
    graph = O.bruteforce_knn(rows, rows, degree, exclude_self=True)[0]
    up = hip.DeviceArray.from_numpy
    sp, d, d_q = O.search_params(64, degree), up(rows), up(rows_of(rng, nq, dim))
    rest = up(graph), up(np.arange(n, dtype=np.uint32)), up(np.zeros(1, np.uint32)), up(np.array([5], np.uint32)), up(np.zeros((nq, 1), np.uint32))

    def search():
        ids, dists = hip.DeviceArray((nq, top_k), np.uint32), hip.DeviceArray((nq, top_k), np.float32)
        hip.search_partitions(d, dim, rest[0], degree, rest[1], rest[2], rest[3], 1, d_q, nq, rest[4], top_k, sp["beam"], sp["max_iterations"],
                              sp["min_iterations"], sp["hash_bit"], sp["hash_reset_interval"], 0, ids, dists)
        return ids.numpy(), dists.numpy()

    expect, make, refused = search(), hip.DeviceArray.__init__, []

    def short(self, shape, dtype):
        if np.dtype(dtype).itemsize * np.prod(shape) > n * 128:
            refused.append(shape)
            raise hip.GlideHipError(2, "glide_hip_malloc")
        make(self, shape, dtype)

    monkeypatch.setattr(hip.DeviceArray, "__init__", short)
    got = search()
    assert len(refused) == 1 and all(np.array_equal(a, b) for a, b in zip(expect, got))


@pytest.mark.parametrize("dim,nq,fractions,packs", [(64, 120, 0.0, True), (128, 200, 0.45, True), (128, 200, 0.55, False), (160, 130, 1.0, False), (256, 1300, 0.4, True),
                                                    (100, 2500, 0.6, False), (4, 300, 1.0, False)])
def test_partitions_for_queries_of_fractions(hip, dim, nq, fractions, packs):
    """Rows are packed for queries that search them: not where most of the first queries have other values.  Same results either way."""
    import ctypes as C
    from oracle import oracle as O
    rng = np.random.default_rng(nq)
    n, degree, top_k = 1500, 32, 10
    rows, queries = rows_of(rng, n, dim), rows_of(rng, nq, dim)
    queries[rng.permutation(nq)[:round(fractions * nq)], rng.integers(dim)] += 0.5
    graph = O.bruteforce_knn(rows, rows, degree, exclude_self=True)[0]
    up = hip.DeviceArray.from_numpy
    sp, d, d_q = O.search_params(64, degree), up(rows), up(queries)
    rest = up(graph), up(rng.permutation(n).astype(np.uint32)), up(np.zeros(1, np.uint32)), up(np.array([5], np.uint32)), up(np.zeros((nq, 1), np.uint32))
    u32 = C.c_uint32
    plain = hip._size_fn("glide_hip_search_partitions_workspace_bytes")(u32(nq), u32(1), u32(top_k))
    got = []
    for num in (0, n):
        size = hip._size_fn("glide_hip_search_partitions_rows_workspace_bytes")(u32(nq), u32(1), u32(top_k), u32(num), u32(dim), u32(degree), u32(sp["beam"]))
        assert (size > plain) == (num > 0)
        ws = hip.DeviceArray.full(size // 4, 0xA5A5A5A5)
        ids, dists, cnt = hip.DeviceArray((nq, top_k), np.uint32), hip.DeviceArray((nq, top_k), np.float32), hip.new_counters()
        hip.check(hip.lib().glide_hip_search_partitions_rows(
            *(hip._ptr(v) if not isinstance(v, int) else u32(v) for v in (d, num, dim, rest[0], degree, *rest[1:4], 1, d_q, nq, rest[4], top_k, sp["beam"],
              sp["max_iterations"], sp["min_iterations"], sp["hash_bit"], sp["hash_reset_interval"])), C.c_int(0), hip._ptr(ids), hip._ptr(dists), hip._ptr(ws),
            C.c_size_t(size), hip._ptr(cnt), None), "search")
        hip.synchronize()
        got.append((ids.numpy(), dists.numpy(), hip.read_counters(cnt)))
    assert all(np.array_equal(a, b) for a, b in zip(got[0], got[1]))
    assert (ws.numpy()[plain // 4:] != 0xA5A5A5A5).any() == packs


def test_every_distance(hip):
    """Rows of bytes have whole squared distances below 2^24: the root of every one of them, correctly rounded (as the fp32 kernels'
    sqrtf and numpy's are), and the number itself for the cosine metric."""
    n = 1 << 24
    out, whole = hip.DeviceArray(n, np.float32), np.arange(n, dtype=np.float32)
    for metric, expect in ((0, np.sqrt(whole)), (1, whole)):
        hip.byte_distances(0, n, metric, out)
        hip.synchronize()
        assert np.array_equal(out.numpy(), expect)
    some = np.random.default_rng(1).integers(0, 4096, 4096)
    rows = np.zeros((4096, 4), np.float32)      # and the fp32 kernels' own distances, of some
    rows[:, 0] = some
    dists = hip.DeviceArray(4096, np.float32)
    hip.distance_batch(hip.DeviceArray.from_numpy(rows), hip.DeviceArray.from_numpy(np.zeros_like(rows)), 4096, 4, 0, dists)
    hip.byte_distances(0, n, 0, out)
    hip.synchronize()
    assert np.array_equal(dists.numpy(), out.numpy()[some * some])
    with pytest.raises(hip.GlideHipError):
        hip.byte_distances(1, n, 0, out)
