"""The pool of page-locked result buffers, with an ordinary allocator in the
place of the library's: reuse by size, the bounds on what it keeps and on what the
program holds, a refused allocation, several threads."""
import ctypes
import gc
import threading

import numpy as np
import pytest

from ouxsbli_amd import _abi, _native
from ouxsbli_amd.batch import PinnedPool


class _Lib:
    def __init__(self, refuse=False):
        self.live, self.refuse, self.lock = {}, refuse, threading.Lock()

    def ox_host_alloc(self, n, out):
        if self.refuse:
            return _abi.OX_ENOMEM
        b = ctypes.create_string_buffer(n)
        p = ctypes.cast(out, ctypes.POINTER(ctypes.c_void_p))
        p[0] = ctypes.addressof(b)
        with self.lock:
            self.live[ctypes.addressof(b)] = b
        return _abi.OX_OK

    def ox_host_free(self, p):
        with self.lock:
            del self.live[p.value]


def _pool(monkeypatch, refuse=False, **kw):
    lib = _Lib(refuse)
    monkeypatch.setattr(_native, "load", lambda: lib)
    return PinnedPool(**kw), lib


def test_reuse_and_bounds(monkeypatch):
    pool, lib = _pool(monkeypatch, keep_bytes=1600, out_bytes=3200)
    a = pool.array((2, 100))
    addr = a.ctypes.data
    view = a[1]
    del a
    gc.collect()
    assert pool.array((200,)).ctypes.data != addr  # a view holds the buffer
    view[:] = 1.0
    del view
    gc.collect()
    held = [pool.array((200,)), pool.array((200,))]
    assert all(h.ctypes.data in lib.live for h in held)
    extra = pool.array((200,))  # over what the program may hold
    assert extra.ctypes.data not in lib.live
    del held
    gc.collect()
    assert len(lib.live) == 1  # one kept, one freed


def test_refused_allocation(monkeypatch):
    pool, lib = _pool(monkeypatch, refuse=True)
    a = pool.array((3, 4))
    a[:] = 2.0
    assert a.shape == (3, 4) and a.dtype == np.float64 and not lib.live
    assert pool._out == 0


@pytest.mark.parametrize("threads", [4])
def test_threads(monkeypatch, threads):
    pool, lib = _pool(monkeypatch)
    bad = []

    def work(k):
        for r in range(200):
            a = pool.array((50 + r % 3,))
            a[:] = k
            if not (a == k).all():
                bad.append((k, r))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    gc.collect()
    assert not bad and pool._out == 0
    assert len(lib.live) <= 3 * threads
