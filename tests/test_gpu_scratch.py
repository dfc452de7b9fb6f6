"""Kept scratch blocks: a returned block serves the next taker of a similar size, blocks that are taken never overlap,
also from several threads, the kept bytes stay within their bound, and trim gives them back. Sorts in a row through
kept blocks give the same as the first."""

import ctypes as C
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _alloc(hip, nbytes):
    p = C.c_void_p()
    assert hip._lib.hipcstone_scratch_alloc(C.byref(p), C.c_size_t(nbytes)) == 0
    return p.value


def _free(hip, p):
    assert hip._lib.hipcstone_scratch_free(C.c_void_p(p)) == 0


def _free_bytes(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip._lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # (of the runtime the library is linked to)
    return free.value


def test_scratch_blocks_are_reused_and_given_back(hip):
    hip._lib.hipcstone_scratch_trim()
    hip.device_sync()
    before = _free_bytes(hip)
    a, b = _alloc(hip, 100 * MB), _alloc(hip, 100 * MB)
    assert abs(a - b) >= 100 * MB
    _free(hip, a)
    assert _alloc(hip, 99 * MB) == a  # of a similar size
    c = _alloc(hip, 30 * MB)  # not half as large
    for p in (a, b, c):
        _free(hip, p)
    d = _alloc(hip, 30 * MB)
    assert d == c
    _free(hip, d)
    for p in [_alloc(hip, 300 * MB) for _ in range(5)]:
        _free(hip, p)
    assert before - _free_bytes(hip) <= (1024 + 64) * MB
    hip._lib.hipcstone_scratch_trim()
    assert before - _free_bytes(hip) <= 64 * MB


def test_scratch_from_threads(hip):
    seen, lock, bad = {}, threading.Lock(), []

    def work(k):
        rng = np.random.RandomState(k)
        for _ in range(200):
            n = int(rng.randint(1, 4 * MB))
            p = _alloc(hip, n)
            with lock:
                if any(p < q + m and q < p + n for q, m in seen.items()):
                    bad.append((p, n))
                seen[p] = n
            with lock:
                del seen[p]
            _free(hip, p)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_sorts_through_kept_blocks(hip):
    rng = np.random.RandomState(3)
    for n in (70000, 65000, 1, 70000):
        keys = rng.randint(0, 1 << 28, n).astype(np.uint32)
        x = [rng.rand(n).astype(np.float32) for _ in range(4)]
        d, o = [hip.DeviceArray.from_numpy(a) for a in x], [hip.DeviceArray(n, np.float32) for _ in range(4)]
        k, p = hip.DeviceArray.from_numpy(keys), hip.DeviceArray(n, np.uint32)
        hip.sort_gather(k, p, *d, *o)
        order = np.argsort(keys, kind="stable")
        assert np.array_equal(p.download(), order) and np.array_equal(k.download(), keys[order])
        assert all(np.array_equal(a.download(), b[order]) for a, b in zip(o, x))


def test_a_program_gets_the_kept_memory_back(hip):
    """What a sort leaves in the library's keeping is free for others after scratch_trim()."""
    n = 4_000_000
    k, p = hip.DeviceArray(n, np.uint32), hip.DeviceArray(n, np.uint32)
    k.upload(np.random.RandomState(7).randint(0, 1 << 30, n).astype(np.uint32))
    x, o = ([hip.DeviceArray(n, np.float32) for _ in range(4)] for _ in range(2))
    for d in x:
        d.upload(np.zeros(n, np.float32))
    hip.sort_gather(k, p, *x, *o)  # (the runtime's own memory for kernels of this size stays)
    hip.scratch_trim()
    before = _free_bytes(hip)
    hip.sort_gather(k, p, *x, *o)
    assert before - _free_bytes(hip) > 100 * MB
    hip.scratch_trim()
    for _ in range(100):  # (the driver counts memory that was just in use as free a little later)
        if before - _free_bytes(hip) <= 64 * MB:
            break
        time.sleep(0.02)
    assert before - _free_bytes(hip) <= 64 * MB


def test_a_sort_refused_while_capturing_loses_no_memory(hip):
    """sort_gather synchronizes, which a capture refuses: it raises, nothing runs, and its blocks serve the next call."""
    rng = np.random.RandomState(4)
    n = 5000
    keys = rng.randint(0, 1 << 28, n).astype(np.uint32)
    x = [hip.DeviceArray.from_numpy(rng.rand(n).astype(np.float32)) for _ in range(4)]
    o = [hip.DeviceArray(n, np.float32) for _ in range(4)]
    k, p = hip.DeviceArray.from_numpy(keys), hip.DeviceArray(n, np.uint32)
    hip.sort_gather(k, p, *x, *o)
    order = p.download()
    k.upload(keys)
    s, graph = hip.Stream(), C.c_void_p()
    for _ in range(3):
        print("sort while capturing", flush=True)
        assert hip._lib.hipStreamBeginCapture(C.c_void_p(s.handle), 0) == 0
        with pytest.raises(hip.HipcstoneError):
            hip.sort_gather(k, p, *x, *o, stream=s)
        if hip._lib.hipStreamEndCapture(C.c_void_p(s.handle), C.byref(graph)) == 0 and graph.value:
            assert hip._lib.hipGraphDestroy(graph) == 0
        hip._lib.hipGetLastError()
    hip.sort_gather(k, p, *x, *o)
    assert np.array_equal(p.download(), order) and not hip._Scratch._late
