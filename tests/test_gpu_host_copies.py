"""Host arrays large enough to move in pieces by several threads: odd sizes
come back as they went, also from two host threads sharing one context."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _round_trips(sa, blocks, cells, seed, n=1):
    g = sa.CartesianGrid(cells, blocks, ((0.0, 1.0),) * 3)
    a = sa.GridArray(g)
    rng = np.random.default_rng(seed)
    for _ in range(n):
        host = rng.standard_normal(g.host_shape)
        a.upload(host)
        if not np.array_equal(a.download(), host):
            return False
    return True


@pytest.mark.parametrize("blocks, cells", [((1, 1, 7), (16, 16, 16)), ((3, 2, 2), (17, 19, 33)),
                                           ((5, 5, 7), (16, 16, 16)), ((1, 1, 1), (120, 11, 90))])
def test_round_trip(blocks, cells):
    import spade_amd as sa
    sa.load()
    print(blocks, cells, flush=True)
    assert _round_trips(sa, blocks, cells, 3)


def test_two_threads_one_context():
    import spade_amd as sa
    sa.load()
    sa.default_context()
    ok = [False, False]

    def go(t):
        ok[t] = _round_trips(sa, (4, 4, 2 + t), (16, 16, 16), t, n=4)
    threads = [threading.Thread(target=go, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert ok == [True, True]


@pytest.mark.parametrize("other", ["up", "up_and_down"])
def test_threads_on_arrays_of_one_grid(other):
    """The arrays of a grid share its staging buffer: one host thread downloads
    a large array over and over while another uploads (and downloads) its own."""
    import spade_amd as sa
    g = sa.CartesianGrid((16, 16, 16), (4, 4, 4), ((0.0, 1.0),) * 3)
    rng = np.random.default_rng(7)
    host = [rng.standard_normal(g.host_shape) for _ in range(2)]
    arr = [sa.GridArray(g).upload(h) for h in host]
    ok = [True, True]

    def down():
        for _ in range(12):
            ok[0] = ok[0] and np.array_equal(arr[0].download(), host[0])

    def up_and_down():
        for n in range(12):
            h = host[1] * (1.0 + n)
            arr[1].upload(h)
            if other == "up_and_down":
                ok[1] = ok[1] and np.array_equal(arr[1].download(), h)
    threads = [threading.Thread(target=down), threading.Thread(target=up_and_down)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print(other, ok, flush=True)
    assert ok == [True, True]
    assert np.array_equal(arr[1].download(), host[1] * 12.0)


def test_pinned_destination():
    """A download into memory that is pinned already goes there directly: the
    same values (also at an odd place in the buffer), in less time than pageable
    memory takes, whose pieces pass through pinned slots (0.64 of it at 20 MB)."""
    import ctypes as C
    import time
    import spade_amd as sa
    lib = sa.load()
    g = sa.CartesianGrid((16, 16, 16), (4, 4, 4), ((0.0, 1.0),) * 3)
    host = np.random.default_rng(5).standard_normal(g.host_shape)
    a = sa.GridArray(g).upload(host)
    hip = C.CDLL("libamdhip64.so")
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipHostFree.argtypes = [C.c_void_p]
    mem = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(mem), host.nbytes + 24, 0) == 0
    try:
        pinned = np.ctypeslib.as_array(C.cast(mem, C.POINTER(C.c_double)), shape=(host.size + 3,))
        pinned[:] = 0.0
        plain = np.zeros(host.size)
        best = {}
        for name, out in (("pinned", pinned[3:]), ("pageable", plain)):
            times = []
            for _ in range(20):
                t0 = time.perf_counter()
                assert lib.spd_array_download(a._h, out.ctypes.data_as(C.POINTER(C.c_double))) == 0
                times.append(time.perf_counter() - t0)
            best[name] = min(times)
            assert np.array_equal(out, host.ravel())
        print(best, flush=True)
        assert np.all(pinned[:3] == 0.0)
        assert best["pinned"] < 0.85 * best["pageable"]
    finally:
        hip.hipHostFree(mem)
