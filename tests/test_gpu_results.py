"""The arrays that hold results, and the copy that fills them.

A solver's results are ordinary memory of the program: a forked child has them, and
they can be resized in place.  (Page-locked memory is a shared mapping of the
driver's that is left out of a child.)  The copy goes through four 8 MB slots with a
worker for every 2 MB (none alone), up to eight; the sizes below lie around those steps, and
every result equals the same copy made straight into page-locked memory.
"""
import ctypes
import os
import threading

import numpy as np
import pytest

from ouxsbli_amd import _native, cases, cases2d
from ouxsbli_amd.batch import Batch, PinnedPool
from ouxsbli_amd.cases import CaseSpec
from ouxsbli_amd.solver import Solver
from ouxsbli_amd.solver2d import Solver2D

pytestmark = pytest.mark.gpu

# padded extents, 40 B a cell: 0.04, 1.9, 3.96, 4.04 MB; a slot less and more; five whole slots and a little more; 40.08
SIZES = [(10, 10, 10), (37, 37, 37), (45, 48, 48), (49, 47, 46), (59, 59, 60), (60, 60, 60), (64, 64, 256),
         (64, 64, 257), (103, 101, 101)]


def _spec(n):
    return CaseSpec(nx=n[0], ny=n[1], nz=n[2], order=2, scheme="SLAU", visc="Euler", visc_order=0, tvd="none",
                    slau_variant="HRSLAU2", rk=3, precision="fp64", threshold=0.4, dt=1e-4, Lx=1.0, Ly=1.0, Lz=1.0)


def _field(shape, seed):
    return np.random.default_rng(seed).standard_normal(shape)


def _ordinary(a):
    """The array's pages are the process's own: a child has a copy of them."""
    addr, inside = a.ctypes.data + a.nbytes // 2, False
    for line in open("/proc/self/smaps"):
        w = line.split()
        if "-" in w[0] and not w[0].endswith(":"):
            lo, hi = (int(x, 16) for x in w[0].split("-"))
            inside = lo <= addr < hi
            private = inside and w[1].endswith("p")
        elif inside and w[0] == "VmFlags:":
            return private and "dc" not in w[1:]
    raise AssertionError("no mapping holds the array")


def _child_reads(a):
    want = a.view(np.uint64).sum()  # the bits: a random state's right-hand side holds NaN
    pid = os.fork()
    if pid == 0:
        os._exit(0 if a.view(np.uint64).sum() == want else 1)
    return os.waitpid(pid, 0)[1] == 0


def test_results_are_ordinary_memory():
    spec = _spec((64, 64, 128))
    with Solver(spec) as s:
        s.set_state(np.abs(_field(spec.state_shape(), 1)) + 1.0)
        out = [s.get_state(), s.get_qj(), s.rhs()]
    spec2 = cases2d.os_spec(nx=300, ny=200)
    with Solver2D(spec2) as s:
        s.init_state()
        out.append(s.get_state())
    spec3 = cases.supersonic_tgv_spec(32)
    with Batch(hbm_budget=1 << 30, max_cases=1, pinned_results=False) as b:
        i = b.admit(spec3, cases.tgv_state(spec3), 1)
        b.run(1)
        out.append(b.retire(i))
    assert all(_ordinary(a) and a.flags.owndata for a in out)
    assert all(_child_reads(a) for a in out)


@pytest.mark.parametrize("n", SIZES)
def test_copy_of_results(n):
    spec = _spec(n)
    QJ = _field(spec.state_shape(), sum(n))
    direct = PinnedPool().array(spec.state_shape())
    with Solver(spec) as s:
        s.set_qj(QJ)
        for _ in range(3):
            np.testing.assert_array_equal(s.get_qj(), QJ)
        Q = s.get_state()
        _native.check(s._lib.ox_get_state(s._h, direct.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
        np.testing.assert_array_equal(Q, direct)


def test_copies_of_several_threads():
    """Six copies at once: more than the page-locked slots that are kept."""
    bad = []

    def one(k):
        spec = _spec(SIZES[2 + k])
        QJ = _field(spec.state_shape(), k)
        with Solver(spec) as s:
            s.set_qj(QJ)
            for r in range(6):
                if not np.array_equal(s.get_qj(), QJ):
                    bad.append((k, r))

    ts = [threading.Thread(target=one, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
