"""Large results: where they go and how many helpers they take."""
import ctypes as C
import os
import threading
import time

import numpy as np
import pytest

import tipl_amd
from conftest import smooth_volume

pytestmark = pytest.mark.gpu

SHAPE = (96, 100, 104)  # an 11 MiB field


def _call(ctx, pair, ptr):
    p = ctx.cdm_param()
    rc = tipl_amd.load_library().tiplhip_cdm_level_iterations(ctx.handle, pair[0].handle, pair[1].handle,
                                                              C.byref(p), 1, ptr)
    assert rc == 0


def _pair(ctx, seed):
    It = smooth_volume(SHAPE, seed)
    return ctx.volume(It), ctx.volume(np.roll(It, 1, 2))


def _threads_during(f):
    """The most threads this process had while f ran, over those before it."""
    count = lambda: len(os.listdir("/proc/self/task"))
    stop, most = threading.Event(), [0]

    def watch():
        while not stop.is_set():
            most[0] = max(most[0], count())

    w = threading.Thread(target=watch)
    w.start()
    time.sleep(0.01)
    before = count()
    f()
    stop.set()
    w.join()
    return most[0] - before


def _runtime():
    """The HIP runtime that the library has loaded."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    lib = C.CDLL(path)
    lib.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    lib.hipHostFree.argtypes = [C.c_void_p]
    return lib


def test_pinned_destinations_take_one_transfer(ctx):
    """Memory that the runtime has pinned, from its start and from an odd place in
    it: the pageable result's bytes, and no helper threads."""
    pair = _pair(ctx, 1)
    n = int(np.prod(SHAPE)) * 3
    want = np.empty(n, np.float32)
    _call(ctx, pair, want.ctypes.data)
    hip, p = _runtime(), C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), 4 * (n + 3), 0) == 0
    pinned = np.ctypeslib.as_array((C.c_float * (n + 3)).from_address(p.value))
    for off in (0, 3):
        out = pinned[off:off + n]
        out[:] = 0
        _call(ctx, pair, out.ctypes.data)
        extra = max(_threads_during(lambda: _call(ctx, pair, out.ctypes.data)) for _ in range(20))
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
        assert extra == 0
    assert hip.hipHostFree(p) == 0


def test_copies_of_many_contexts_at_once(ctx):
    """Twelve contexts return results at a time: each its own, with the helper
    threads of four staged copies at most (two each at this size)."""
    pairs = [_pair(ctx, 10 + i) for i in range(12)]
    n = int(np.prod(SHAPE)) * 3
    want = [np.empty(n, np.float32) for _ in pairs]
    got = [np.empty(n, np.float32) for _ in pairs]
    for p, w in zip(pairs, want):
        _call(ctx, p, w.ctypes.data)
    others = [tipl_amd.Context(0) for _ in pairs]
    for c, p, g in zip(others, pairs, got):  # (streams and code objects are there)
        _call(c, p, g.ctypes.data)

    def run():
        t = [threading.Thread(target=lambda c=c, p=p, g=g: [_call(c, p, g.ctypes.data) for _ in range(10)])
             for c, p, g in zip(others, pairs, got)]
        for x in t:
            x.start()
        for x in t:
            x.join()

    for g in got:
        g[:] = 0
    extra = _threads_during(run)
    for g, w in zip(got, want):
        assert np.array_equal(g.view(np.uint32), w.view(np.uint32))
    for c in others:
        c.close()
    assert extra <= len(pairs) + 4 * 2
