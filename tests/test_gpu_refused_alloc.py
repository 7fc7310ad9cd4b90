"""A refused allocation is reported once, by the call that asked for it.

HIP keeps the error of a refused allocation until it is read; the launch check of
the next call must not find it.  The sizes below are over every address space, so
the host's allocator refuses them before anything is reserved.
"""
import ctypes

import numpy as np
import pytest

from ouxsbli_amd import _abi, _native, cases, cases2d
from ouxsbli_amd.batch import PinnedPool
from ouxsbli_amd.solver import Solver
from ouxsbli_amd.solver2d import Solver2D

pytestmark = pytest.mark.gpu

TOO_LARGE = 1 << 60


def _refuse():
    p = ctypes.c_void_p()
    assert _native.load().ox_host_alloc(TOO_LARGE, ctypes.byref(p)) != _abi.OX_OK
    assert not p.value


def test_refused_host_allocation_leaves_no_error():
    spec = cases.supersonic_tgv_spec(16)
    with Solver(spec) as s:
        s.set_state(cases.tgv_state(spec))
        _refuse()
        s.step(1)
        _refuse()
        Q = s.get_state()
        _refuse()
        R = s.rhs()
    assert np.isfinite(Q).all() and np.isfinite(R).all()
    spec2 = cases2d.os_spec(nx=40, ny=30)
    with Solver2D(spec2) as s:
        s.init_state()
        _refuse()
        s.step(1)
        _refuse()
        assert np.isfinite(s.get_state()).all()


def test_result_of_a_refused_page_lock():
    """The pool's fallback: an ordinary array, which the next call fills."""
    pool = PinnedPool()
    lib = pool._lib

    class Refusing:
        def ox_host_alloc(self, n, out):
            return lib.ox_host_alloc(TOO_LARGE, out)

    pool._lib = Refusing()
    spec = cases.supersonic_tgv_spec(16)
    with Solver(spec) as s:
        s.set_state(cases.tgv_state(spec))
        s.step(1)
        Q = pool.array(spec.state_shape())
        _native.check(lib.ox_get_state(s._h, Q.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
        np.testing.assert_array_equal(Q, s.get_state())
