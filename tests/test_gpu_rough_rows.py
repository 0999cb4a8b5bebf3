"""Sub-graph builds and refinement that look at rows in fp16 first, against the same calls without the fp16 copy: the copy
only says which rows need not be measured, so graphs and counters must agree to the bit.  The rows include equal ones, near ties
far below fp16's resolution, values at the ends of fp32's range, and values that are infinite or none."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INV = 0xFFFFFFFF


@pytest.fixture(scope="module")
def hip():
    from glide_amd import capi
    capi.set_device(0)
    return capi


def rows_of(rng, n, dim, kind):
    x = rng.standard_normal((6, dim))[rng.integers(0, 6, n)] * 0.5 + rng.standard_normal((n, dim)) * 0.3
    if kind == "unit":
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    elif kind == "whole":            # equal distances
        x = np.rint(x * 2)
    elif kind == "close":            # far from the origin: fp16 tells few of them apart
        x = 40 + x * 0.01
    elif kind == "spread":           # most values far below what fp16 holds next to the largest
        x[:, 1:] *= 1e-4
        x[:: 50, 0] = 3e4
    elif kind == "tiny":
        x *= 1e-21
    elif kind == "huge":
        x *= 3e17
    x[n // 2: n // 2 + 8] = x[3]
    x = x.astype(np.float32)
    if kind == "infinite":
        x[n // 3, 5] = np.inf
    elif kind == "nan":
        x[n // 3, dim - 1] = np.nan
    return x


def packed(hip, rows):
    d = hip.DeviceArray.from_numpy(rows)
    n, dim = rows.shape
    d_rough = hip.DeviceArray(hip.rough_rows_bytes(n, dim), np.uint8)
    hip.pack_rough_rows(d, n, dim, d_rough)
    return d, d_rough


@pytest.mark.parametrize("n,dim,kind", [(1, 516, "plain"), (90, 4, "unit"), (65, 100, "close"), (300, 1024, "spread"), (77, 960, "tiny"), (77, 960, "huge"), (40, 600, "nan")])
def test_packed_rows(hip, n, dim, kind):
    rows = rows_of(np.random.default_rng(n), max(n, 16), dim, kind)[:n]
    held = packed(hip, rows)[1].numpy()
    most = held[:4].view(np.uint32)[0]
    assert most == np.abs(rows).view(np.uint32).max()
    if kind == "nan":
        return
    unit = np.float64(2.0) ** (max(int(most >> 23), 14) - 127 - 13)
    rounded = held[256:].view(np.float16).reshape(n, (dim + 7) // 8 * 8).astype(np.float64) * unit
    assert not rounded[:, dim:].any()
    rounded = rounded[:, :dim]
    # half a unit in the eleventh place, or the smallest normal number where numbers below it are dropped
    assert (np.abs(rounded - rows) <= np.maximum(np.abs(rows.astype(np.float64)) * 2.0 ** -11, 2.0 ** -14 * unit)).all()


def test_lengths_that_are_not_held(hip):
    assert hip.rough_rows_bytes(100, 1028) == 0 and hip.rough_rows_bytes(100, 514) == 0 and hip.rough_rows_bytes(100, 0) == 0
    assert hip.rough_rows_bytes(100, 516) == 256 + 100 * 520 * 2
    d = hip.DeviceArray((4, 1028), np.float32)
    with pytest.raises(hip.GlideHipError):
        hip.pack_rough_rows(d, 4, 1028, hip.DeviceArray(16384, np.uint8))


@pytest.mark.parametrize("dim,knn_degree,degree,build_beam,refine_beam,metric,relaxant,kind", [
    (4, 16, 8, 32, 64, 0, 1.05, "plain"), (28, 32, 32, 64, 128, 0, 1.05, "unit"), (96, 32, 32, 128, 64, 1, 1.05, "unit"), (128, 64, 48, 64, 128, 0, 1.05, "plain"),
    (128, 32, 32, 64, 64, 1, 1.05, "whole"), (132, 32, 32, 64, 64, 0, 1.05, "spread"), (200, 32, 24, 128, 128, 1, 1.05, "unit"), (256, 32, 32, 64, 64, 0, 1.05, "close"),
    (260, 32, 64, 64, 128, 0, 1.05, "huge"), (384, 48, 48, 128, 64, 1, 1.05, "tiny"), (512, 32, 32, 64, 64, 0, 1.05, "nan"), (512, 64, 32, 64, 128, 0, 1.1, "plain"),
    (516, 16, 8, 32, 64, 0, 1.05, "plain"), (960, 32, 32, 64, 128, 0, 1.05, "plain"), (960, 64, 32, 128, 96, 1, 1.05, "unit"), (1024, 32, 64, 96, 64, 1, 1.2, "unit"),
    (768, 32, 32, 64, 128, 0, 1.0, "whole"), (640, 64, 24, 128, 128, 1, 0.9, "whole"), (960, 32, 32, 64, 64, 0, 1.05, "close"), (960, 32, 32, 128, 64, 1, 1.05, "close"),
    (520, 32, 32, 64, 128, 0, 1.05, "spread"), (960, 32, 32, 64, 64, 0, 1.05, "tiny"), (960, 32, 32, 64, 64, 1, 1.05, "tiny"), (960, 32, 32, 64, 64, 0, 1.05, "huge"),
    (960, 32, 32, 64, 64, 1, 1.05, "huge"), (800, 32, 32, 64, 64, 0, 1.05, "infinite"), (800, 32, 32, 64, 128, 1, 1.05, "nan"), (960, 32, 32, 64, 64, 0, 0.0, "plain")])
def test_build_and_refine(hip, dim, knn_degree, degree, build_beam, refine_beam, metric, relaxant, kind):
    from oracle import oracle as O
    rng = np.random.default_rng(dim + degree + metric)
    lengths, boundary = (400, 300), 120
    n = sum(lengths)
    rows = rows_of(rng, n, dim, kind)
    reorder = np.concatenate([rows, rows[rng.permutation(n)[:boundary]]])
    mp = np.concatenate([rng.permutation(n), rng.permutation(n)[:boundary]]).astype(np.uint32)
    starts, lens = np.array([0, lengths[0], n], np.uint32), np.array([*lengths, boundary], np.uint32)
    finite = np.nan_to_num(reorder, nan=0.0, posinf=0.0) * np.float32({"tiny": 1e21, "huge": 1e-17}.get(kind, 1))
    knn = np.concatenate([O.bruteforce_knn(finite[s:s + m], finite[s:s + m], knn_degree, metric, exclude_self=True)[0] for s, m in zip(starts, lens)])
    knn[:, knn_degree // 2:] = rng.integers(0, boundary, knn[:, knn_degree // 2:].shape)     # and rows that are far away
    knn[rng.random(knn.shape) < 0.05] = INV
    b, r = O.search_params(build_beam, knn_degree), O.search_params(refine_beam, max(knn_degree, degree))
    d_re, d_re_rough = packed(hip, reorder)
    d_rows, d_rows_rough = packed(hip, rows)
    up = hip.DeviceArray.from_numpy
    d_knn, d_map, d_s, d_l = up(knn), up(mp), up(starts), up(lens)
    d_sp, d_c, d_gsp = up(np.array([5, 9, 2], np.uint32)), up(rows[[20, 600]] + np.float32(0.25)), up(np.array([3, 500], np.uint32))
    got = []
    for re_rough, row_rough in ((None, None), (d_re_rough, d_rows_rough)):
        g, out, cnt = hip.DeviceArray.full((n, degree), INV), hip.DeviceArray.full((n, degree), 0xDEADBEEF), hip.new_counters()
        args = (b["beam"], b["max_iterations"], b["min_iterations"], b["hash_bit"], b["hash_reset_interval"], relaxant, metric, g, cnt)
        hip.build_subgraph(d_re, n, dim, d_knn, knn_degree, d_map, d_s, d_l, 3, d_sp, degree, *args, rough_rows=re_rough)
        hip.build_boundary(d_re, n, n + boundary, dim, d_knn, knn_degree, d_map, 2, degree, *args, rough_rows=re_rough)
        hip.refine(d_rows, n, dim, g, out, degree, d_c, 2, d_gsp, r["beam"], r["max_iterations"], r["min_iterations"], r["hash_bit"],
                   r["hash_reset_interval"], relaxant, metric, cnt, order=d_map, rough_rows=row_rough)
        hip.synchronize()
        got.append((g.numpy(), out.numpy(), hip.read_counters(cnt)))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]
    assert (got[0][1] != INV).any()


@pytest.mark.parametrize("dim,degree,knn_degree,metric", [(96, 32, 32, 1), (160, 48, 64, 0), (128, 24, 72, 0), (960, 64, 64, 0), (1028, 32, 32, 0)])
def test_whole_build(hip, monkeypatch, dim, degree, knn_degree, metric):
    """The same index with and without the copy, also where only one of its stages takes it or none does."""
    from glide_amd import index as G
    rows = rows_of(np.random.default_rng(dim), 3000, dim, "unit" if metric == 1 else "plain")
    graphs = []
    for pays in (False, True):
        monkeypatch.setattr(G, "rough_rows_pay", lambda num, dim, pays=pays: pays)
        d = hip.DeviceArray.from_numpy(rows)
        d_reorder, d_map, starts, lengths, d_c = G.preprocess(G.PartitionParameter(centroid_num=3, boundary_factor=1.04, sample_factor=0.5, metric=metric), d)
        d_knn = G.build_nnd(G.NNDescentParameter(graph_degree=knn_degree, max_iterations=6), d_reorder, starts, lengths)
        index = G.GLIDE(degree, d, d_c, metric)
        index.build(G.IndexParameter(graph_degree=degree, knn_degree=knn_degree, relaxant_factor=1.05, metric=metric),
                    G.make_search_parameter(64, knn_degree), G.make_search_parameter(128, max(knn_degree, degree)), d_knn, starts, lengths, d_map, d_reorder)
        graphs.append(index.d_graph.numpy())
    assert np.array_equal(*graphs) and (graphs[0] != INV).mean() > 0.5


def test_where_it_pays():
    from glide_amd.index import rough_rows_pay as pays
    assert pays(60_000, 960) and pays(250_000, 128) and pays(1_000_000, 96)
    assert not pays(2_000, 512) and not pays(70_000, 128) and not pays(234_567, 96) and not pays(10_000_000, 64)


def survey(rows, turn, tiny, graph, starts, lengths, start_points):
    """glide_hip_survey_rough_rows in numpy: [far neighbours of neighbours, those told, rows, rows whose walk goes astray]."""
    n, counts = len(rows), [0, 0, 0, 0]
    x = rows.astype(np.float64)
    for row in np.arange(min(n, 256)) * n // min(n, 256):
        seg = np.flatnonzero((row >= starts) & (row < starts + lengths.astype(np.int64)))
        if len(seg) == 0:
            continue
        first, length = int(starts[seg[0]]), int(lengths[seg[0]])

        def neighbours(of):
            ids = graph[first + of, :32].astype(np.int64)
            ids = ids[(ids < length) & (ids != row - first)]
            return ids, np.linalg.norm(x[first + ids] - x[row], axis=1)

        ids, d = neighbours(row - first)
        if len(ids) == 0:
            continue
        other, e = neighbours(ids[len(ids) // 2])
        far = ~np.isin(other, ids) & (e >= d.max())
        told = far & (e * (1 - 2 * 4.93e-4) - 2 * turn * np.linalg.norm(x[row]) - tiny >= d.max())
        at, nearest = int(start_points[seg[0]]) if start_points[seg[0]] < length else 0, np.inf
        while True:
            there, f = neighbours(at)
            if len(there) == 0 or f.min() >= nearest:
                break
            at, nearest = int(there[f.argmin()]), f.min()
        counts = [counts[0] + far.sum(), counts[1] + told.sum(), counts[2] + 1, counts[3] + (not nearest <= 1.5 * d.max())]
    return [int(c) for c in counts]


@pytest.mark.parametrize("n,dim,degree,kind", [(1, 8, 4, "plain"), (40, 4, 3, "plain"), (700, 128, 32, "unit"), (600, 132, 64, "close"), (513, 260, 20, "plain"),
                                               (900, 512, 72, "unit"), (511, 960, 40, "plain"), (640, 1024, 16, "close")])
def test_survey(hip, n, dim, degree, kind):
    from oracle import oracle as O
    rng = np.random.default_rng(n)
    rows = rows_of(rng, max(n, 16), dim, kind)[:n]
    starts, lengths = np.array([0, n // 3, n // 3], np.uint32), np.array([n // 3, 0, n - n // 3], np.uint32)
    graph = np.full((n, degree), INV, np.uint32)
    for s, m in zip(starts, lengths):
        k = min(degree, m - 1) if m else 0
        if k > 0:
            graph[s:s + m, :k] = O.bruteforce_knn(rows[s:s + m], rows[s:s + m], k, exclude_self=True)[0]
    graph[rng.random(graph.shape) < 0.1] = INV
    start_points = np.array([max(n // 3 - 1, 0), 0, 1 << 30], np.uint32)
    d, d_rough = packed(hip, rows)
    head = d_rough.numpy()[:8]
    unit = np.float64(2.0) ** (max(int(head[:4].view(np.uint32)[0] >> 23), 14) - 127 - 13)
    d_counts = hip.DeviceArray(4, np.uint32)
    hip.survey_rough_rows(d, d_rough, n, dim, hip.DeviceArray.from_numpy(graph), degree, hip.DeviceArray.from_numpy(starts),
                          hip.DeviceArray.from_numpy(lengths), 3, hip.DeviceArray.from_numpy(start_points), d_counts)
    got, expect = [int(v) for v in d_counts.numpy()], survey(rows, float(head[4:].view(np.float32)[0]), np.sqrt(dim) * 3 * 6.2e-5 * unit, graph, starts, lengths, start_points)
    # a comparison of two sums of squares can go the other way where they agree to (dim + 8) 2^-24: less than one in ten thousand here
    assert got[2] == expect[2] and all(abs(g - e) <= 2 + 1e-3 * expect[0] for g, e in zip(got, expect)), (got, expect)


@pytest.mark.parametrize("metric,degree,knn_degree", [(0, 32, 32), (1, 32, 32), (0, 32, 72)])
@pytest.mark.parametrize("kind", ["plain", "dense", "apart"])
def test_a_copy_that_tells_nothing_is_not_used(hip, monkeypatch, kind, metric, degree, knn_degree):
    """Clusters so dense that rounding blurs them, and clusters so far apart that searches end in the wrong one: the builds do without the
    copy.  Rows of low intrinsic dimension: they take it.  (72 neighbours a row: the sub-graphs never take it, refinement decides by itself.)"""
    from glide_amd import index as G
    rng = np.random.default_rng(8)
    n, dim = 6000, 96
    if kind == "plain":
        rows = rng.standard_normal((n, 6)) @ rng.standard_normal((6, dim)) + rng.standard_normal((n, dim)) * 0.1
    else:
        rows = rng.random((12, dim))[rng.integers(0, 12, n)] * 160 + rng.standard_normal((n, dim)) * (0.05 if kind == "dense" else 8)
    rows = rows.astype(np.float32)
    taken, graphs = [], []
    for name in ("build_subgraph", "build_boundary", "refine"):
        def spy(*args, call=getattr(hip, name), **kw):
            taken.append(kw["rough_rows"] is not None)
            return call(*args, **kw)
        monkeypatch.setattr(hip, name, spy)
    for pays in (True, False):
        monkeypatch.setattr(G, "rough_rows_pay", lambda num, dim, pays=pays: pays)
        d = hip.DeviceArray.from_numpy(rows)
        d_reorder, d_map, starts, lengths, d_c = G.preprocess(G.PartitionParameter(centroid_num=3, boundary_factor=1.04, sample_factor=0.5, metric=metric), d)
        d_knn = G.build_nnd(G.NNDescentParameter(graph_degree=knn_degree, max_iterations=8), d_reorder, starts, lengths)
        index = G.GLIDE(degree, d, d_c, metric)
        index.build(G.IndexParameter(graph_degree=degree, knn_degree=knn_degree, relaxant_factor=1.05, metric=metric),
                    G.make_search_parameter(64, knn_degree), G.make_search_parameter(128, knn_degree), d_knn, starts, lengths, d_map, d_reorder)
        graphs.append(index.d_graph.numpy())
        if pays:
            assert taken[-1] == (kind == "plain") and not any(taken[:-1]) == (kind != "plain" or knn_degree > 64), taken
        else:
            assert not any(taken)
        taken.clear()
    assert np.array_equal(*graphs)
