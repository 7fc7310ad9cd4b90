"""Launch shapes of the FP32-bulk sweeps.

On a uniform periodic grid every cell takes the same operations, so a field that is
moved by a few cells gives the moved result, bit for bit, wherever the seams of the
x sweep's runs and rows, of the y and z sweeps' groups and segments and of the
boundary fill come to lie: a value that a seam got wrong would not move with the
field.  Between walls the field moves along the periodic directions.  The sizes are
the smallest grids, widths around a wave's, a workgroup's and a run's cells, whole
rows of 64 and 128 cells, and row counts around groups of four.
"""
import dataclasses

import numpy as np
import pytest

from ouxsbli_amd import cases
from ouxsbli_amd.batch import Batch
from ouxsbli_amd.solver import Solver
from oracle_lib import Oracle
from test_gpu_parity import _perturbed_tgv, _spec

pytestmark = pytest.mark.gpu

SCHEMES = {
    "slau6-ns6-rk3": (6, "SLAU", "NS", 6, "hybrid", "HRSLAU2", 3),
    "hybrid6-me4-rk3": (6, "Hybrid", "NS", 6, "hybrid", "HRSLAU2", 3, "ME4Base"),
    "keep4-ns4-rk4": (4, "KEEP", "NS", 4, "none", "HRSLAU2", 4),
    "keep4-euler-rk4": (4, "KEEP", "Euler", 0, "none", "HRSLAU2", 4),
    "roe2-euler-rk3": (2, "Roe", "Euler", 0, "none", "HRSLAU2", 3),
}
SIZES = [(12, 37, 12), (62, 33, 12), (63, 13, 14), (64, 17, 15), (65, 66, 13), (126, 14, 65), (128, 19, 13),
         (252, 13, 12), (254, 17, 12)]
SHIFT = (7, 5, 3)  # cells along x, y, z


def _moved(Q, order, dirs):
    """The interior moved along `dirs`, ghost layers filled again (periodic)."""
    h = order // 2
    M = Q.copy()
    M[h:-h, h:-h, :, h:-h] = np.roll(Q[h:-h, h:-h, :, h:-h], [SHIFT[d] for d in dirs], [(3, 1, 0)[d] for d in dirs])
    return cases.periodic_fill(M, order)


def _run(spec, Q, steps=2):
    with Solver(spec) as s:
        s.set_state(Q)
        s.step(steps)
        return s.get_state()


@pytest.mark.parametrize("name", list(SCHEMES))
@pytest.mark.parametrize("n", SIZES)
def test_fp32_result_moves_with_the_field(name, n):
    spec = dataclasses.replace(_spec(*SCHEMES[name], n=n, Ma=0.6), precision="fp32_bulk")
    Q = _perturbed_tgv(spec)
    print(f"fp32 shapes {name} {n}", flush=True)
    a = _run(spec, Q)
    assert np.isfinite(a).all() and np.abs(a - Q).max() > 0
    np.testing.assert_array_equal(_run(spec, _moved(Q, spec.order, (0, 1, 2))), _moved(a, spec.order, (0, 1, 2)))


@pytest.mark.parametrize("bc", [("periodic", "slip", "periodic"), ("slip", "periodic", "extrapolate"),
                                ("periodic", "periodic", "slip")], ids="-".join)
@pytest.mark.parametrize("name", ["hybrid6-me4-rk3", "keep4-ns4-rk4"])
def test_fp32_between_walls_moves_with_the_field(name, bc):
    spec = dataclasses.replace(_spec(*SCHEMES[name], n=(65, 29, 30), Ma=0.6), precision="fp32_bulk", bc=bc)
    dirs = [d for d in range(3) if bc[d] == "periodic"]
    h = spec.order // 2
    sl = (slice(h, -h), slice(h, -h), slice(None), slice(h, -h))

    def filled(Q):
        o = Oracle(spec)
        o.set_qj(Q)
        o.set_bc()
        return o.get_qj()

    Q = filled(_perturbed_tgv(spec))
    a = _run(spec, Q)
    assert np.isfinite(a).all() and np.abs(a - Q).max() > 0
    b = _run(spec, filled(_moved(Q, spec.order, dirs)))
    np.testing.assert_array_equal(b[sl], _moved(a, spec.order, dirs)[sl])


def test_fp32_batched_equals_alone():
    specs = [dataclasses.replace(_spec(*SCHEMES["slau6-ns6-rk3"], n=n, Ma=0.6), precision="fp32_bulk") for n in SIZES]
    Q = [_perturbed_tgv(s) for s in specs]
    with Batch(hbm_budget=4 << 30, max_cases=len(specs), autotune=False) as b:
        ids = [b.admit(s, q, 2) for s, q in zip(specs, Q)]
        b.run(2)
        got = {i: b.retire(i) for i in b.done()}
    for i, s, q in zip(ids, specs, Q):
        np.testing.assert_array_equal(got[i], _run(s, q))
