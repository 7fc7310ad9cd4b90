"""The longest 2-D grid that is accepted, as thin as it may be: 8 x 2^27 points.

Its 19 million tiles of 512 lanes and its 2^32 state values are more work items
than one dimension of a launch takes.  The oblique-shock state differs from row to
row at the two ends only, and the spacings are powers of two, so every row away
from the ends equals the oracle's on a grid of 64 rows, and the ends equal its
ends, bit for bit.
"""
import ctypes

import numpy as np
import pytest

from ouxsbli_amd import _abi, cases2d
from ouxsbli_amd._native import OxError
from ouxsbli_amd.solver2d import Solver2D
from oracle_lib import Oracle2D

pytestmark = pytest.mark.gpu

NX, NY, END = 8, 1 << 27, 32
_libc = ctypes.CDLL(None)
_libc.memcmp.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]


def _spec(ny):
    h = 2.0 ** -10
    return cases2d.os_spec(nx=NX, ny=ny, Lx=h * (NX - 1), Ly=h * (ny - 1), dt=2.0 ** -22)


def _check(Q, ref):
    """The ends, and each row between them equal to the next."""
    np.testing.assert_array_equal(Q[:END], ref[:END])
    np.testing.assert_array_equal(Q[-END:], ref[-END:])
    row = Q[0].nbytes
    a = Q.ctypes.data + (END - 1) * row
    assert _libc.memcmp(a, a + row, (NY - 2 * END + 1) * row) == 0


def test_longest_strip_matches_oracle_rows():
    try:
        import psutil
        if psutil.virtual_memory().available < 80 << 30:
            pytest.skip("needs 80 GiB of free host memory")
    except ImportError:
        pass
    small = _spec(2 * END)
    with Solver2D(small) as s:  # (the device's state, as for the strip: fewer than 10 columns split nowhere)
        s.init_state()
        Q0 = s.get_state()
    o = Oracle2D(small)
    o.set_state(Q0)
    o.step(1)
    ref = o.get_state()
    # the premise: the rows in the middle are alike, and the ends have moved
    assert np.array_equal(ref[END - 8:END + 8], np.broadcast_to(ref[END], (16,) + ref[END].shape))
    assert np.abs(ref - Q0).max() > 0

    try:
        s = Solver2D(_spec(NY))
    except OxError as e:
        if e.code == _abi.OX_ENOMEM:
            pytest.skip("needs 103 GB of device memory")
        raise
    with s:
        print(f"strip {NX} x {NY}", flush=True)
        s.init_state()
        s.step(1)
        print("stepped", flush=True)
        Q = s.get_state()
        print("read", flush=True)
        _check(Q, ref)
        s.init_state()
        s.set_state(Q)
        print("written", flush=True)
        Q[:] = 0.0
        Q = s.get_state()
        _check(Q, ref)
