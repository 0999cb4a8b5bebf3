"""k-means kernels at the sizes where their layouts change: rows of up to 128 dims (half a wavefront a row) and beyond,
samples that pass through LDS while seeding (32768 rows) and one row more, sums in LDS (4096 values) and in memory, and
samples that do not fill a workgroup.  Integer rows: every distance and every sum is exact, so the outcome is one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_of(n, dim, seed):
    return np.random.default_rng(seed).integers(0, 16, (n, dim)).astype(np.float32)


@pytest.mark.parametrize("n, dim, k", [(1, 4, 1), (63, 128, 3), (65, 132, 5), (1000, 256, 9), (200, 260, 4), (32768, 8, 3), (32769, 8, 3), (32770, 132, 40), (33000, 260, 12)])
def test_seeding_rows(n, dim, k):
    from glide_amd import capi as hip
    from oracle import oracle as O
    hip.set_device(0)
    x = rows_of(n, dim, n)
    e_cent, e_rows = O.kmeans_seed(x, k, 5)
    cent, rows = hip.DeviceArray((k, dim), np.float32), hip.DeviceArray(k, np.uint32)
    sb = hip.kmeans_seed_workspace_bytes(n)
    ws = hip.DeviceArray(sb // 8 + 1, np.uint64)
    hip.kmeans_seed(hip.DeviceArray.from_numpy(x), n, dim, k, 5, cent, ws, sb, chosen_rows=rows)
    hip.synchronize()
    assert np.array_equal(rows.numpy(), e_rows)
    assert np.array_equal(cent.numpy(), e_cent)


@pytest.mark.parametrize("n, dim, k", [(1, 4, 1), (31, 128, 32), (129, 128, 32), (300, 128, 33), (257, 100, 5), (1000, 4, 256), (900, 132, 7)])
def test_one_lloyd_step(n, dim, k):
    from glide_amd import capi as hip
    hip.set_device(0)
    x = rows_of(n, dim, 3 * n + k)
    start = rows_of(k, dim, k)          # equal distances are common: the first centroid wins
    cent = hip.DeviceArray.from_numpy(start)
    wb = hip.kmeans_workspace_bytes(k, dim)
    ws = hip.DeviceArray(wb // 8 + 1, np.uint64)
    hip.kmeans_fit(hip.DeviceArray.from_numpy(x), n, dim, k, 1, cent, ws, wb)
    hip.synchronize()
    nearest = ((x[:, None].astype(np.float64) - start[None]) ** 2).sum(-1).argmin(1)
    expect = start.copy()
    for c in range(k):
        if (nearest == c).any():
            expect[c] = (x[nearest == c].sum(0, dtype=np.float64) / (nearest == c).sum()).astype(np.float32)
    assert np.array_equal(cent.numpy(), expect)


# one side and the other of every line between the two kernels of a Lloyd step: sums in LDS (up to 16, 64 and 1024 clusters)
# and in memory
@pytest.mark.parametrize("n, dim, k", [(499, 4, 1), (500, 4, 1), (1199, 128, 8), (1201, 100, 8), (2000, 28, 16), (4250, 128, 17), (4249, 128, 17),
                                       (16001, 64, 64), (22100, 60, 65), (22099, 60, 65), (348160, 4, 1024), (11999, 128, 33), (12000, 128, 33),
                                       (12003, 100, 256)])
def test_one_lloyd_step_by_either_kernel(n, dim, k):
    from glide_amd import capi as hip
    hip.set_device(0)
    x, start = rows_of(n, dim, n + k), rows_of(k, dim, k)
    cent = hip.DeviceArray.from_numpy(start)
    wb = hip.kmeans_workspace_bytes(k, dim)
    ws = hip.DeviceArray(wb // 8 + 1, np.uint64)
    hip.kmeans_fit(hip.DeviceArray.from_numpy(x), n, dim, k, 1, cent, ws, wb)
    hip.synchronize()
    half = (start ** 2).sum(1) / 2                                       # integers and halves below 2^24: exact
    nearest = np.concatenate([(half - x[i:i + 4096] @ start.T).argmin(1) for i in range(0, n, 4096)])
    sums, counts = np.zeros((k, dim)), np.bincount(nearest, minlength=k)
    np.add.at(sums, nearest, x)
    expect = np.where(counts[:, None] > 0, sums / np.maximum(counts, 1)[:, None], start).astype(np.float32)
    assert np.array_equal(cent.numpy(), expect)


# few points beside the size of the centroids, and many beside it: the scratch of the fit is larger than that of the draw of the sample, and smaller
@pytest.mark.parametrize("num, dim, parts", [(1000, 960, 16), (3000, 128, 256), (10_000, 1000, 200), (60_000, 28, 5)])
def test_partitioning_whatever_scratch_is_largest(num, dim, parts):
    from glide_amd import capi as hip
    from glide_amd import index as G
    hip.set_device(0)
    x = rows_of(num, dim, num)
    param = G.PartitionParameter(centroid_num=parts, boundary_factor=1.04, sample_factor=0.1, metric=G.Metric.Euclidean)
    d_reorder, d_map, starts, lengths, d_centroids = G.preprocess(param, hip.DeviceArray.from_numpy(x))
    # the centroids: the steps one at a time, each with the scratch that it asks for
    sample = x[np.random.default_rng(param.seed).permutation(num)[:max(num // 10, parts)]]
    d_sample, cent = hip.DeviceArray.from_numpy(sample), hip.DeviceArray((parts, dim), np.float32)
    size = hip.kmeans_seed_workspace_bytes(len(sample))
    hip.kmeans_seed(d_sample, len(sample), dim, parts, param.seed, cent, hip.DeviceArray(size // 8 + 1, np.uint64), size)
    size = hip.kmeans_workspace_bytes(parts, dim)
    hip.kmeans_fit(d_sample, len(sample), dim, parts, param.kmeans_iterations, cent, hip.DeviceArray(size // 8 + 1, np.uint64), size)
    hip.synchronize()
    assert np.array_equal(d_centroids.numpy(), cent.numpy())
    assert int(lengths[:parts].sum()) == num
    assert np.array_equal(d_reorder.numpy(), x[d_map.numpy()])
