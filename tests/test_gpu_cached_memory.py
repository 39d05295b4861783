"""The buffers kept from destroyed H-matrices: they serve the next ones, stay within their
bounds (4096 buffers and 4 GiB per device), and go back when asked for."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _cached(gpu):
    out = (ctypes.c_int64 * 6)()
    gpu.lib().hmg_cached_memory(out)
    return {"bytes": out[0], "blocks": out[1], "large_bytes": out[2], "pinned_bytes": out[4], "pinned": out[5]}


def _build(gpu, kern, n, dim, k=12):
    X = O.uniform(71 + n, dim * n).reshape(dim, n)
    hm = gpu.HMatrix(X, X, 32 if dim == 2 else 20, 1.0, 50, 64, k)
    hm.setup()
    hm.set_kernel(kern)
    hm.precompute_aca()
    return hm


def test_kept_buffers_serve_the_next_h_matrix(gpu):
    gpu.lib().hmg_release_cached_memory()
    assert _cached(gpu)["blocks"] == 0 and _cached(gpu)["bytes"] == 0
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 0.1)
    x = O.normal(72, 6000)
    hm = _build(gpu, kern, 6000, 3)
    first = hm.apply(x)
    hm.destroy()
    kept = _cached(gpu)
    assert kept["blocks"] > 10 and kept["bytes"] > 8 * 6000 * 12
    hm = _build(gpu, kern, 6000, 3)
    np.testing.assert_array_equal(hm.apply(x), first)
    held = _cached(gpu)
    assert held["blocks"] < kept["blocks"] // 2 and held["bytes"] < kept["bytes"] // 2
    hm.destroy()
    # the same buffers came back
    assert _cached(gpu)["blocks"] <= kept["blocks"] + 4
    gpu.lib().hmg_release_cached_memory()
    assert _cached(gpu)["blocks"] == 0 and _cached(gpu)["bytes"] == 0
    kern.free()


def test_kept_buffers_stay_within_their_bounds(gpu):
    gpu.lib().hmg_release_cached_memory()
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 0.1)
    most = 0
    hms = [_build(gpu, kern, 2000 + i, 2) for i in range(300)]
    for hm in hms:
        hm.destroy()
        most = max(most, _cached(gpu)["blocks"])
        assert most <= 4096
    assert most == 4096  # reached (some 16 buffers each): the oldest went for the last ones
    hms = [_build(gpu, kern, n, 3, k=24) for n in (60000, 50000, 40000)]
    for hm in hms:
        hm.destroy()
        assert _cached(gpu)["blocks"] <= 4096 and _cached(gpu)["bytes"] <= 4 << 30
    assert _cached(gpu)["bytes"] > 2 << 30
    gpu.lib().hmg_release_cached_memory()
    assert _cached(gpu)["blocks"] == 0
    kern.free()


def test_staging_buffers_of_ended_threads(gpu):
    # more worker threads than buffers may wait: those past the bound are freed by the next
    # thread that takes one, and none is lost
    import threading

    from hmglib_amd import hip
    n_threads = 90
    x = np.arange(64, dtype=np.float64)
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 0.1)
    X = O.uniform(73, 2 * 600).reshape(2, 600)

    def at_once(count):
        hms = [gpu.HMatrix(X, X, 32, 1.0, 50, 64, 8) for _ in range(count)]
        gate = threading.Barrier(count)

        def work(hm):
            gate.wait()
            hm.setup()  # stages copies through the thread's buffer
            gate.wait()

        ts = [threading.Thread(target=work, args=(hm,)) for hm in hms]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for hm in hms:
            hm.destroy()

    gpu.lib().hmg_release_cached_memory()
    assert _cached(gpu)["pinned"] == 0
    at_once(n_threads)
    assert _cached(gpu)["pinned"] == n_threads
    at_once(1)
    assert _cached(gpu)["pinned"] <= 65
    for _ in range(3):
        at_once(n_threads)
    at_once(1)
    assert _cached(gpu)["pinned"] <= 65
    gpu.lib().hmg_release_cached_memory()
    assert _cached(gpu)["pinned"] == 0 and _cached(gpu)["pinned_bytes"] == 0
    d = hip.DeviceArray(x)
    np.testing.assert_array_equal(d.download(), x)
    d.free()
    kern.free()
