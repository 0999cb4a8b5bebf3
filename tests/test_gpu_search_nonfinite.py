"""Beam search where distances are not finite: rows and queries with a NaN, rows so far away that the distance overflows.

A row whose distance is not a number is no candidate beside rows that have one, in any degree or beam bucket, so a search
over such rows must give, bit for bit, what the oracle gives on the same graph with the edges to them removed.  A query
with a NaN has nothing else: it gets neighbours of its entry point.  Infinite distances are ordered and must come out as
the oracle's networks leave them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INV, NO_ROW = 0xFFFFFFFF, 0x7FFFFFFF
DEGREES = [24, 32, 64, 96, 128, 160, 256]


@pytest.fixture(scope="module")
def hip():
    from glide_amd import capi
    capi.set_device(0)
    return capi


def _index(seed, n, dim, deg, centroid_num):
    rng = np.random.default_rng(seed)
    data = rng.integers(0, 9, (n, dim)).astype(np.float32)             # exact sums, ties
    queries = rng.integers(0, 9, (24, dim)).astype(np.float32)
    graph = np.stack([rng.permutation(n)[:deg] for _ in range(n)]).astype(np.uint32)
    centroids = data[rng.permutation(n)[:centroid_num]].copy()
    return rng, data, queries, graph, centroids, rng.permutation(n)[:centroid_num].astype(np.uint32)


@pytest.mark.parametrize("dim", [32, 320])
@pytest.mark.parametrize("deg", DEGREES)
def test_rows_with_nan_beside_others(hip, deg, dim):
    from oracle import oracle as O
    from test_gpu_search import run_gpu_search
    rng, data, queries, graph, centroids, start_points = _index(deg + dim, 1500, dim, deg, 5)
    bad = rng.random(data.shape[0]) < 0.2
    bad[start_points] = False
    data[bad, rng.integers(0, dim, int(bad.sum()))] = np.nan
    without = np.where(bad[graph], np.uint32(INV), graph)
    for beam in (32, 48, 64, 128, 160, 256, 288, 512):
        sp = O.search_params(beam, deg)
        print("degree", deg, "dim", dim, "beam", beam, flush=True)
        eids, edists, est = O.search(np.nan_to_num(data), without, centroids, start_points, queries, min(beam, 64), **sp)
        gids, gdists, gcnt = run_gpu_search(hip, data, graph, centroids, start_points, queries, min(beam, 64), sp, counters=True)
        assert np.array_equal(gids, eids) and np.array_equal(gdists, edists)
        assert (gcnt[0], gcnt[2]) == (est["iterations"], est["graph_rows"])


@pytest.mark.parametrize("dim", [32, 320])
@pytest.mark.parametrize("deg", DEGREES)
def test_entry_among_rows_with_nan(hip, deg, dim):
    """All neighbours of the entry point have a NaN and lead to one and the same row of neighbours, most of them finite: the
    search goes on from there, whatever the degree and beam, as if it had started at one of them."""
    from oracle import oracle as O
    from test_gpu_search import run_gpu_search
    rng, data, queries, graph, centroids, start_points = _index(deg + dim + 1, 1500, dim, deg, 1)
    row = graph[start_points[0]]
    row[row == start_points[0]] = np.setdiff1d(np.arange(data.shape[0]), row)[0]     # the entry is not its own neighbour
    first = row.copy()
    bad = rng.random(data.shape[0]) < 0.1
    bad[first] = True
    bad[start_points[0]] = False
    data[bad] = np.nan
    onward = rng.permutation(np.flatnonzero(~bad))[:deg]
    onward[: deg // 4] = np.flatnonzero(bad)[: deg // 4]
    graph[first] = onward
    without = np.where(bad[graph], np.uint32(INV), graph)
    for beam in (32, 64, 128, 160, 256, 288, 512):
        sp = O.search_params(beam, deg)
        sp.update(max_iterations=2000, hash_bit=13, hash_reset_interval=4000)   # one visited set throughout: the phase of its resets is not the point
        print("degree", deg, "dim", dim, "beam", beam, flush=True)
        eids, edists, _ = O.search(np.nan_to_num(data), without, centroids, first[:1].copy(), queries, min(beam, 64), **sp)
        gids, gdists, _ = run_gpu_search(hip, data, graph, centroids, start_points, queries, min(beam, 64), sp)
        assert np.array_equal(gids, eids) and np.array_equal(gdists, edists)


@pytest.mark.parametrize("dim", [32, 320])
@pytest.mark.parametrize("deg", DEGREES)
def test_query_with_nan(hip, deg, dim):
    from oracle import oracle as O
    from test_gpu_search import run_gpu_search
    _, data, queries, graph, centroids, start_points = _index(deg + dim + 2, 1500, dim, deg, 40)
    asked = queries.copy()
    asked[::2, 3] = np.nan
    for beam in (32, 64, 128, 160, 256, 288, 512):
        top_k = min(beam, 64)
        sp = O.search_params(beam, deg)
        print("degree", deg, "dim", dim, "beam", beam, flush=True)
        eids, edists, _ = O.search(data, graph, centroids, start_points, queries, top_k, **sp)
        gids, gdists, _ = run_gpu_search(hip, data, graph, centroids, start_points, asked, top_k, sp)
        assert np.array_equal(gids[1::2], eids[1::2]) and np.array_equal(gdists[1::2], edists[1::2])   # the queries beside them
        got, near = gids[::2], graph[start_points[0]]       # the first centroid: none is nearer to such a query
        row = got != NO_ROW
        assert np.isin(got[row], near).all() and np.isnan(gdists[::2][row]).all() and row[:, 0].all()
        if deg in (64, 128, 256):                           # no empty slots: nothing but rows
            assert row[:, : min(deg, top_k)].all()


@pytest.mark.parametrize("deg", [24, 32, 48, 64, 96, 160])
def test_rows_at_infinite_distance(hip, deg):
    from oracle import oracle as O
    from test_gpu_search import run_gpu_search
    rng, data, queries, graph, centroids, start_points = _index(deg + 7, 1500, 32, deg, 5)
    far = rng.random(data.shape[0]) < 0.6
    far[start_points] = False
    data[far, 1] = 3e30                                     # its square is infinite
    for beam in (48, 64, 96, 128, 256, 288, 512):
        for iterations in (2, 3, 5, 400):                   # also the beams early on, which still hold such rows
            sp = O.search_params(beam, deg)
            sp["max_iterations"] = iterations
            print("degree", deg, "beam", beam, "iterations", iterations, flush=True)
            eids, edists, _ = O.search(data, graph, centroids, start_points, queries, beam, **sp)
            gids, gdists, _ = run_gpu_search(hip, data, graph, centroids, start_points, queries, beam, sp)
            assert np.array_equal(gids, eids) and np.array_equal(gdists, edists)
