"""Device memory that freed arrays leave for later ones: reuse, its bounds, what freeing promises, threads."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture()
def hip():
    from glide_amd import capi
    capi.set_device(0)
    capi.release_memory()
    yield capi
    capi.release_memory()


def address(d):
    return d._address


def test_reuse_by_size(hip):
    a = hip.DeviceArray(10 << 20, np.uint8)
    at = address(a)
    a.free()
    assert address(hip.DeviceArray(11 << 20, np.uint8)) != at             # too small
    assert address(hip.DeviceArray(7 << 20, np.uint8)) != at              # more than a fifth of it would be idle
    b = hip.DeviceArray(9 << 20, np.uint8)
    assert address(b) == at
    with pytest.raises(hip.GlideHipError):                                # a block that is freed twice is not handed out twice
        b.free()
        hip.check(hip.lib().glide_hip_free(hip.vp(at)), "glide_hip_free")
    assert address(hip.DeviceArray(10 << 20, np.uint8)) == at


def test_held_memory_counts_as_free_and_is_bounded(hip):
    before, slack = hip.mem_info()[0], 64 << 20      # the device hands out memory in pieces of some MiB
    arrays = [hip.DeviceArray(600 << 20, np.uint8) for _ in range(5)]
    assert hip.mem_info()[0] < before - (2500 << 20)
    for d in arrays:
        d.free()
    assert abs(hip.mem_info()[0] - before) <= slack
    hip.release_memory()
    assert abs(hip.mem_info()[0] - before) <= slack
    huge = hip.DeviceArray((2 << 30) + 4096, np.uint8)                     # never held
    huge.free()
    assert abs(hip.mem_info()[0] - before) <= slack


def test_work_has_ended_when_free_returns(hip):
    """A block goes to its next owner, on another stream, while the kernels of the last one would still write it."""
    streams = []
    for _ in range(2):
        s = hip.vp()
        hip.check(hip.lib().glide_hip_stream_create(hip.C.byref(s)), "glide_hip_stream_create")
        streams.append(s)
    s1, s2 = (s.value for s in streams)
    n = 16 << 20
    src = hip.DeviceArray.full((n // 128, 128), 7)
    hip.synchronize()
    for _ in range(5):
        a = hip.DeviceArray((n // 128, 128), np.uint32)
        for _ in range(20):
            hip.copy_rows(src, n // 128, 128, a, 128, stream=s1)
        at = address(a)
        a.free()
        b = hip.DeviceArray((n // 128, 128), np.uint32)
        assert address(b) == at
        hip.check(hip.lib().glide_hip_fill_u32(hip.vp(at), hip.u32(3), hip.C.c_size_t(n), hip.vp(s2)), "fill")
        hip.synchronize(s2)
        hip.synchronize(s1)
        assert (b.numpy() == 3).all()
        b.free()
    for s in streams:
        hip.check(hip.lib().glide_hip_stream_destroy(s), "glide_hip_stream_destroy")


def test_threads(hip):
    errors = []

    def work(seed):
        rng = np.random.default_rng(seed)
        try:
            for _ in range(60):
                n = int(rng.integers(1, 1 << 18))
                d = hip.DeviceArray.full(n, seed)
                if not (d.numpy() == seed).all():
                    errors.append(seed)
                d.free()
        except Exception as e:      # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not errors
