"""The k-means sample drawn on the device: the first entries of numpy's permutation for the same seed, around the sizes where a
chunk of draws ends (16 384 draws, some 1.4 for every id) and where ids gain a bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num", [1, 2, 3, 5, 64, 1000, 8192, 8193, 11_000, 16_385, 32_768, 65_537, 200_003, 1_000_000])
def test_the_permutation_of_the_seed(num):
    from glide_amd import capi as hip
    hip.set_device(0)
    wb = hip.sample_ids_workspace_bytes(num)
    ws = hip.DeviceArray.full(wb // 16 * 4 + 4, 0xDEADBEEF)
    for seed in (7, 0, 123_456_789):
        expect = np.random.default_rng(seed).permutation(num)
        for count in sorted({1, max(1, num // 100), num}):
            ids = hip.DeviceArray.full(count, 0xDEADBEEF)
            hip.sample_ids(num, count, seed, ids, ws, wb)
            hip.synchronize()
            assert np.array_equal(ids.numpy(), expect[:count]), (seed, count)


def test_bad_arguments():
    from glide_amd import capi as hip
    hip.set_device(0)
    wb = hip.sample_ids_workspace_bytes(100)
    ws, ids = hip.DeviceArray(wb // 16 + 1, np.dtype("V16")), hip.DeviceArray(101, np.uint32)
    for num, count, size in ((0, 0, wb), (100, 101, wb), (100, 10, wb - 1)):
        with pytest.raises(hip.GlideHipError):
            hip.sample_ids(num, count, 7, ids, ws, size)


def test_partitioning_where_the_device_does_not_draw(monkeypatch):
    """More rows than the device draws from, or no memory for its scratch: the host draws the same sample."""
    from glide_amd import capi as hip
    from glide_amd import index as G
    hip.set_device(0)
    assert hip.sample_ids_workspace_bytes(1 << 30) > 0 and hip.sample_ids_workspace_bytes((1 << 30) + 1) == 0
    x = np.random.default_rng(1).integers(0, 256, (20_000, 32)).astype(np.float32)
    param = G.PartitionParameter(centroid_num=8, boundary_factor=1.04, sample_factor=0.05, metric=G.Metric.Euclidean)
    got = []
    for size in (hip.sample_ids_workspace_bytes, lambda num: 0, lambda num: 1 << 46):
        with monkeypatch.context() as m:
            m.setattr(hip, "sample_ids_workspace_bytes", size)
            d_reorder, d_map, starts, lengths, d_centroids = G.preprocess(param, hip.DeviceArray.from_numpy(x))
        got.append((d_reorder.numpy(), d_map.numpy(), starts, lengths, d_centroids.numpy()))
    for other in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got[0], other))
