"""Tile shapes of the 2-D stage on the GPU.

A launch takes tiles of 64 x 3 cells where the device holds them all at once and
of 64 x 7 otherwise (a small case among many in a batch).  The interiors below are
whole tiles and one cell less or more in each direction; every FP64 state equals
the CPU oracle bit for bit, and both heights give the same FP32 bits.
"""
import numpy as np
import pytest

from ouxsbli_amd import cases2d as c2
from ouxsbli_amd.batch import Batch
from ouxsbli_amd.solver2d import Solver2D
from oracle_lib import Oracle2D
from test_gpu_2d import noisy_os_state

pytestmark = pytest.mark.gpu

SIZES = [(66, 23), (65, 24), (67, 25), (130, 9), (131, 10), (46, 44)]
# 1333 and 16 x 342 tiles of 3 rows: more than the 1024 workgroups that fit at most
LARGE = [(66, 4000), (1026, 1028)]


def _spec(n, precision="fp64", scheme="SLAU", order=6):
    return c2.os_spec(nx=n[0], ny=n[1], scheme=scheme, order=order, precision=precision, cfl=0.3)


def _oracle(spec, Q, steps):
    o = Oracle2D(spec)
    o.set_state(Q)
    o.step(steps)
    return o.get_state()


@pytest.mark.parametrize("scheme,order", [("SLAU", 6), ("Roe", 4), ("SLAU", 2)])
@pytest.mark.parametrize("n", SIZES + LARGE)
def test_2d_tiles_bitwise(n, scheme, order):
    spec = _spec(n, scheme=scheme, order=order)
    Q = noisy_os_state(spec, 3)
    print(f"2-D tiles {scheme} {order} {n}", flush=True)
    steps = 3 if n in SIZES else 1
    with Solver2D(spec) as s:
        s.set_state(Q)
        s.step(steps)
        got = s.get_state()
    np.testing.assert_array_equal(got, _oracle(spec, Q, steps))


@pytest.mark.parametrize("precision", ["fp64", "fp32_bulk"])
def test_2d_small_cases_in_tall_tiles(precision):
    """Small cases beside a large one of their kind: 7 rows instead of 3."""
    specs = [_spec(n, precision) for n in SIZES + LARGE[1:]]
    Q = [noisy_os_state(s, k) for k, s in enumerate(specs)]
    with Batch(hbm_budget=4 << 30, max_cases=len(specs), autotune=False) as b:
        ids = [b.admit(s, q, 2) for s, q in zip(specs, Q)]
        b.run(2)
        got = {i: b.retire(i) for i in b.done()}
    for i, s, q in zip(ids, specs, Q):
        with Solver2D(s) as alone:
            alone.set_state(q)
            alone.step(2)
            np.testing.assert_array_equal(got[i], alone.get_state())
