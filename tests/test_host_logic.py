"""Host-side logic of the product that needs no GPU: parameter arithmetic, file formats, datasets."""
import numpy as np

from glide_amd import datasets as D
from glide_amd import index as G
from oracle import oracle as O


def test_parameter_arithmetic_matches_reference_restatement():
    for beam in (1, 31, 32, 33, 50, 64, 100, 128, 200, 256, 300, 512):
        for degree in (16, 32, 64, 96, 128, 256):
            mi, b = G.adjust_search_params(0, 0, beam)
            assert (mi, b) == O.adjust_search_params(0, 0, beam)
            hb = G.calculate_hash_bitlen(b, degree, 0.5, 0)
            assert hb == O.hash_bitlen(b, degree, 0.5, 0)
            assert G.calculate_hash_reset_interval(b, degree, 0.5, hb) == O.hash_reset_interval(b, degree, 0.5, hb)
    assert G.adjust_search_params(90, 0, 64) == O.adjust_search_params(90, 0, 64)
    assert G.adjust_search_params(0, 500, 70) == O.adjust_search_params(0, 500, 70)
    p = G.make_search_parameter(50, 32)
    assert (p.beam, p.max_iterations, p.hash_bit, p.hash_reset_interval) == (64, 56, 8, 2)   # test.sh search beam 50
    assert G.NNDescentParameter(graph_degree=32).intermediate_graph_degree == 48


def test_unsupported_sizes_raise_like_the_reference():
    import pytest
    with pytest.raises(ValueError, match="Unsupported beam"):
        G._check_sizes(513, 32)
    with pytest.raises(ValueError, match="Unsupported beam"):
        G._check_sizes(300, 32)        # above 256 a beam is a multiple of 16; adjust_search_params never hands out another
    for beam in (1, 50, 255, 256, 288, 320, 448, 480, 512):
        G._check_sizes(beam, 32)
    assert all(G.adjust_search_params(0, 0, b)[1] % 32 == 0 for b in range(1, 513))
    with pytest.raises(ValueError, match="Unsupported graph_degree"):
        G._check_sizes(64, 257)


def test_seeding_workspace_holds_what_is_used():
    """Distances to the candidates (32 bytes a row) are kept for samples whose steps pass through LDS, 32768 rows; a larger
    sample needs its smallest distances and 8 potentials per 64 rows."""
    from glide_amd import capi
    size = capi.kmeans_seed_workspace_bytes
    assert size(32768) >= 36 * 32768
    for n in (32769, 50_000, 1_000_001):
        assert 4 * n + 64 * (n // 64) <= size(n) <= 4 * n + 64 * (n // 64 + 1) + 512


def test_file_formats_round_trip(tmp_path):
    rng = np.random.default_rng(0)
    m = rng.standard_normal((7, 5)).astype(np.float32)
    D.write_fbin(tmp_path / "m.fbin", m)
    raw = np.fromfile(tmp_path / "m.fbin", dtype=np.uint32)
    assert raw[0] == 7 and raw[1] == 5 and raw.size == 2 + 35           # u32 num, u32 dim, rows
    assert np.array_equal(D.read_fbin(tmp_path / "m.fbin"), m)
    g = rng.integers(0, 100, (4, 3)).astype(np.uint32)
    D.write_fbin(tmp_path / "g", g)
    assert np.array_equal(D.read_fbin(tmp_path / "g", np.uint32), g)
    D.write_vector(tmp_path / "v", [3, 1, 4])
    assert np.fromfile(tmp_path / "v", dtype=np.uint32).tolist() == [3, 3, 1, 4]
    assert D.read_vector(tmp_path / "v").tolist() == [3, 1, 4]
    D.write_segment(tmp_path / "s", [0, 10, 30], [10, 20, 5])
    assert np.fromfile(tmp_path / "s", dtype=np.uint32).tolist() == [3, 0, 10, 30, 10, 20, 5]   # n, starts, lengths
    s, l = D.read_segment(tmp_path / "s")
    assert s.tolist() == [0, 10, 30] and l.tolist() == [10, 20, 5]


def test_synthetic_generators_are_seeded_and_shaped():
    a, b = D.gmm_clipped(1000, 128, seed=5), D.gmm_clipped(1000, 128, seed=5)
    assert np.array_equal(a, b) and a.dtype == np.float32
    assert a.min() >= 0 and a.max() <= 255 and np.array_equal(a, np.rint(a))
    assert not np.array_equal(a, D.gmm_clipped(1000, 128, seed=6))
    c = D.gmm_normalized(500, 96)
    assert np.allclose(np.linalg.norm(c, axis=1), 1, atol=1e-5)
    e = D.beta_scaled(200, 960)
    assert e.shape == (200, 960) and e.min() >= 0 and e.max() <= 1
    r = D.recall(np.array([[1, 2, 3]]), np.array([[3, 4, 1]]), 3)
    assert abs(r - 2 / 3) < 1e-9


def test_copies_that_only_save_time_never_fail_a_call(monkeypatch):
    """Short memory, memory that is gone when it is asked for, and more rows than are packed: no copy, no error."""
    import pytest
    from glide_amd import capi
    asked = []

    class NoMemory:
        def __init__(self, shape, dtype):
            if np.dtype(dtype) == np.uint8:
                asked.append(shape)
                raise capi.GlideHipError(code, "glide_hip_malloc")

    class Rows:
        shape = (100_000, 256)

    code = 2                 # hipErrorOutOfMemory
    monkeypatch.setattr(capi, "DeviceArray", NoMemory)
    monkeypatch.setattr(capi, "mem_info", lambda: (1 << 40, 1 << 40))
    assert G.spare_array(1 << 20) is None and G.byte_rows(Rows()) is None and G.rough_rows(Rows()) is None
    assert len(asked) == 3
    code = 719               # another error is none of memory
    with pytest.raises(capi.GlideHipError):
        G.spare_array(1 << 20)
    monkeypatch.setattr(capi, "mem_info", lambda: (1 << 20, 1 << 40))
    assert G.spare_array((1 << 19) + 1) is None
    # 2^32 pieces of 16 bytes are packed at most
    for dim, most in ((4, 2 ** 29), (128, 2 ** 29), (132, 2 ** 28), (256, 2 ** 28)):
        assert capi.byte_rows_bytes(most, dim) == 2 ** 36 and capi.byte_rows_bytes(most + 1, dim) == 0
        plain = capi._size_fn("glide_hip_search_partitions_workspace_bytes")(64, 8, 10)
        size = capi._size_fn("glide_hip_search_partitions_rows_workspace_bytes")
        assert size(64, 8, 10, 100, dim, 32, 64) > plain and size(2 ** 31, 8, 10, most + 1, dim, 64, 512) == capi._size_fn("glide_hip_search_partitions_workspace_bytes")(2 ** 31, 8, 10)


def test_a_search_beside_one_that_lets_the_byte_rows_go():
    """Two threads search an index whose rows have become known to others: both find that the copy may not be used."""
    class Rows:
        writes, shared = 3, True

    class Index(G.GLIDE):
        reads = 0

        @property
        def _bytes(self):      # held when this thread looks, gone a moment later
            self.reads += 1
            return (object(), self.d_data, 3) if self.reads == 1 else None

        @_bytes.setter
        def _bytes(self, value):
            assert value is None

    index = Index.__new__(Index)
    index.d_data = Rows()
    assert index._byte_rows() is None
