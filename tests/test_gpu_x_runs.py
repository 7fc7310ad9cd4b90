"""Launch shapes of the x sweep on the GPU.

The faces of a band of 8 to 32 rows follow one another; a workgroup takes 253 of
them, the last shared with the next workgroup, a wave 64, the last shared with
the next wave.  The widths below are the smallest grids (many rows in one
workgroup), rows of about one wave's and one workgroup's faces and of more, and row
counts that leave a shorter last band; every right-hand side equals the CPU
oracle bit for bit (the FP64 kernels round every operation as the oracle does).
"""
import numpy as np
import pytest

from ouxsbli_amd.batch import Batch
from ouxsbli_amd.solver import Solver
from oracle_lib import Oracle
from test_gpu_parity import _perturbed_tgv, _spec

pytestmark = pytest.mark.gpu

SCHEMES = {
    "slau6-ns6-rk3": (6, "SLAU", "NS", 6, "hybrid", "HRSLAU2", 3),
    "keep4-euler-rk4": (4, "KEEP", "Euler", 0, "none", "HRSLAU2", 4),
    "hybrid2-euler-rk3": (2, "Hybrid", "Euler", 0, "hybrid", "HRSLAU2", 3),
    "hybrid6-les-rk4": (6, "Hybrid", "LES", 6, "hybrid", "HRSLAU2", 4),
}
SIZES = [(12, 13, 12), (62, 33, 12), (63, 35, 13), (65, 12, 12), (125, 17, 12), (126, 14, 12), (250, 13, 12),
         (251, 12, 13), (252, 19, 12), (254, 14, 12), (505, 12, 12)]


def _oracle(spec, Q, steps):
    o = Oracle(spec)
    o.set_state(Q)
    o.step(steps)
    return o.get_state()


@pytest.mark.parametrize("name", list(SCHEMES))
@pytest.mark.parametrize("n", SIZES)
def test_x_runs_bitwise(name, n):
    spec = _spec(*SCHEMES[name], n=n, Ma=0.6)
    Q = _perturbed_tgv(spec)
    print(f"x runs {name} {n}", flush=True)
    with Solver(spec) as s:
        s.set_state(Q)
        s.step(1)
        got = s.get_state()
    np.testing.assert_array_equal(got, _oracle(spec, Q, 1))


def test_x_runs_batched_bitwise():
    specs = [_spec(*SCHEMES["slau6-ns6-rk3"], n=n, Ma=0.6) for n in SIZES]
    Q = [_perturbed_tgv(s) for s in specs]
    with Batch(hbm_budget=4 << 30, max_cases=len(specs), autotune=False) as b:
        ids = [b.admit(s, q, 1) for s, q in zip(specs, Q)]
        b.run(1)
        got = {i: b.retire(i) for i in b.done()}
    for i, s, q in zip(ids, specs, Q):
        np.testing.assert_array_equal(got[i], _oracle(s, q, 1))
