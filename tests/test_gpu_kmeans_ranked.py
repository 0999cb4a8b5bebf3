"""Lloyd steps whose nearest centroids are ranked on the matrix cores: the sizes where that kernel takes over, its tiles' edges,
centroids too close to rank and rows whose norms overflow."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def one_step(x, start):
    from glide_amd import capi as hip
    hip.set_device(0)
    (n, dim), k = x.shape, len(start)
    cent = hip.DeviceArray.from_numpy(start)
    wb = hip.kmeans_workspace_bytes(k, dim)
    ws = hip.DeviceArray(wb // 8 + 1, np.uint64)
    hip.kmeans_fit(hip.DeviceArray.from_numpy(x), n, dim, k, 1, cent, ws, wb)
    hip.synchronize()
    return cent.numpy()


def means(x, start, nearest):
    k = len(start)
    sums, counts = np.zeros(start.shape), np.bincount(nearest, minlength=k)
    np.add.at(sums, nearest, x.astype(np.float64))
    return np.where(counts[:, None] > 0, sums / np.maximum(counts, 1)[:, None], start)


# one side and the other of the rule, tiles of 128 points and 32 centroids with remainders, up to 256 centroids and one more
@pytest.mark.parametrize("n, dim, k", [(1999, 128, 64), (2000, 128, 64), (2001, 100, 65), (2111, 68, 255), (2176, 128, 256), (2176, 128, 257), (2000, 256, 128),
                                       (5999, 132, 16), (6000, 132, 16), (6001, 960, 33), (2003, 1000, 200)])
def test_integer_rows(n, dim, k):
    rng = np.random.default_rng(n + k)
    x, start = (rng.integers(0, 8, (m, dim)).astype(np.float32) for m in (n, k))
    start[k // 2] = start[1]                                             # equal distances: the first centroid wins
    half = (start.astype(np.float64) ** 2).sum(1) / 2
    nearest = (half - x.astype(np.float64) @ start.T.astype(np.float64)).argmin(1)
    assert np.array_equal(one_step(x, start), means(x, start, nearest).astype(np.float32))


@pytest.mark.parametrize("dim, k", [(128, 100), (320, 40)])
def test_centroids_too_close_to_rank(dim, k):
    """A dozen centroids a few rounding errors apart, far from zero; rows whose nearest two differ by less than the fp32 sums
    can tell are left out, so one answer is right."""
    rng = np.random.default_rng(dim)
    start = rng.normal(0, 1, (k, dim)) + 30.0
    start[5:17] = start[5] + rng.normal(0, 3e-3, (12, dim))
    start = start.astype(np.float32)
    x = (start[rng.integers(0, k, 9000)] + rng.normal(0, 0.05, (9000, dim))).astype(np.float32)
    d = np.stack([((x.astype(np.float64) - c) ** 2).sum(1) for c in start.astype(np.float64)], 1)
    two = np.sort(d, 1)[:, :2]
    x, d = x[two[:, 1] - two[:, 0] > 1e-4 * two[:, 1]], d[two[:, 1] - two[:, 0] > 1e-4 * two[:, 1]]
    assert len(x) > 6000 and (np.sort(d, 1)[:, 5] - np.sort(d, 1)[:, 0] < 0.1).mean() > 0.02
    got, expect = one_step(x, start), means(x, start, d.argmin(1))
    assert np.abs(got - expect).max() < 1e-5                             # fp32 means of values near 30: half a unit is 1e-6


def test_norms_that_overflow():
    """|x|^2 is infinite where |x - c|^2 is not: the nearest centroid is found all the same."""
    rng = np.random.default_rng(1)
    k, dim = 64, 128
    start = rng.normal(0, 1, (k, dim)).astype(np.float32)
    start[40:] = (rng.choice([-1.0, 1.0], (k - 40, dim)) * 4e18).astype(np.float32)
    x = (start[rng.integers(40, k, 2500)] * (1 + rng.normal(0, 1e-3, (2500, dim)))).astype(np.float32)
    d = np.stack([((x.astype(np.float64) - c) ** 2).sum(1) for c in start.astype(np.float64)], 1)
    assert (d.min(1) < 1e38).all() and ((x.astype(np.float64) ** 2).sum(1) > 4e38).all()
    got, expect = one_step(x, start), means(x, start, d.argmin(1))
    assert np.abs(got - expect).max() <= 1e-6 * np.abs(expect).max()
