"""The SGS viscosity's walk of eight planes, with ragged ends.

A workgroup takes 32 x 8 columns of the computed cells (all but the outermost
layer) and walks eight planes of them where that leaves 512 workgroups or more, four
otherwise.  This grid takes the walk of eight with one column over in x and in y and
a last walk of seven planes; its right-hand side and its state after a step equal
the CPU oracle bit for bit.
"""
import numpy as np
import pytest

from ouxsbli_amd.solver import Solver
from oracle_lib import Oracle
from test_gpu_parity import _perturbed_tgv, _spec

pytestmark = pytest.mark.gpu

N = (125, 125, 123)


def test_les_walk_of_eight_planes_bitwise():
    spec = _spec(6, "Hybrid", "LES", 6, "hybrid", "HRSLAU2", 4, n=N, Ma=0.5)
    cx, cy, cz = spec.nx - 2, spec.ny - 2, spec.nz - 2  # computed cells
    assert (cx % 32, cy % 8, cz % 8) == (1, 1, 7)
    assert -(-cx // 32) * -(-cy // 8) * -(-cz // 8) >= 512
    Q = _perturbed_tgv(spec)
    o = Oracle(spec)
    o.set_state(Q)
    h = spec.order // 2
    sl = (slice(h, -h), slice(h, -h), slice(None), slice(h, -h))
    print("oracle", flush=True)
    Ro = o.rhs()
    o.step(1)
    with Solver(spec) as s:
        s.set_state(Q)
        np.testing.assert_array_equal(s.rhs()[sl], Ro[sl])
        s.step(1)
        np.testing.assert_array_equal(s.get_state(), o.get_state())
