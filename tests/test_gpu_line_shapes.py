"""Launch shapes of the y and z sweeps on the GPU: the segment lengths chosen
from the grid, and the y sweep's runs across rows.

The y sweep runs through the cells of one group of four z rows after another in
workgroups of 64 cells, and both sweeps are cut into segments whose length
depends on the grid and on the other cases of a batch.  The interiors below are
the smallest grids, widths around the workgroup's 64 cells, and row counts
around the groups of four; every result equals the CPU oracle bit for bit (the
FP64 kernels round every operation as the oracle does).
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
    "keep4-ns4-rk4": (4, "KEEP", "NS", 4, "none", "HRSLAU2", 4),
    "roe2-euler-rk3": (2, "Roe", "Euler", 0, "none", "HRSLAU2", 3),
}
SIZES = [(12, 12, 12), (63, 13, 14), (64, 12, 15), (65, 17, 12), (129, 14, 13), (20, 66, 65)]


def _run(spec, Q, steps):
    o = Oracle(spec)
    o.set_state(Q)
    o.step(steps)
    return o.get_state()


@pytest.mark.parametrize("name", list(SCHEMES))
@pytest.mark.parametrize("n", SIZES)
def test_line_shapes_bitwise(name, n):
    spec = _spec(*SCHEMES[name], n=n, Ma=0.6)
    Q = _perturbed_tgv(spec)
    print(f"line shapes {name} {n}", flush=True)
    with Solver(spec) as s:
        s.set_state(Q)
        s.step(2)
        got = s.get_state()
    np.testing.assert_array_equal(got, _run(spec, Q, 2))


def test_line_shapes_batched_bitwise():
    """Uneven cases that share launches, and lengths, then one of them alone."""
    specs = [_spec(*SCHEMES["slau6-ns6-rk3"], n=n, Ma=0.6) for n in SIZES]
    steps = [1, 1, 2, 1, 3, 1]
    Q = [_perturbed_tgv(s) for s in specs]
    got = {}
    with Batch(hbm_budget=4 << 30, max_cases=len(specs), autotune=False) as b:
        ids = [b.admit(s, q, k) for s, q, k in zip(specs, Q, steps)]
        while b.run(8)[1]:
            pass
        for i in b.done():
            got[i] = b.retire(i)
    for i, s, q, k in zip(ids, specs, Q, steps):
        np.testing.assert_array_equal(got[i], _run(s, q, k))
