"""When a batch tunes segment lengths: for a case that is admitted into a group of
its own, not for one that shares launches, whose lengths are chosen for all of
them together.

Tuning evaluates up to nine lengths, four right-hand sides each (21 ms at 160^3),
where an admission without it takes half a millisecond, so the admission times tell
which were tuned.
"""
import time

import numpy as np
import pytest

from ouxsbli_amd import cases
from ouxsbli_amd.batch import Batch
from ouxsbli_amd.solver import Solver

pytestmark = pytest.mark.gpu

SIZES = (152, 160, 156)


def _specs(precision="fp64"):
    return [cases.supersonic_tgv_spec(n, precision=precision) for n in SIZES]


def _admit(b, spec):
    t = time.perf_counter()
    cid = b.admit(spec, None, 1)
    return cid, time.perf_counter() - t


def test_admission_tunes_only_a_case_alone_in_its_group():
    specs = _specs()
    with Batch(hbm_budget=32 << 30, max_cases=8, autotune=False) as b:  # (loads the kernels)
        plain = [_admit(b, s)[1] for s in specs + specs][3:]
    with Batch(hbm_budget=32 << 30, max_cases=8, autotune=True) as b:
        alone = _admit(b, specs[0])[1]
        shared = [_admit(b, s)[1] for s in specs[1:]]
        other = _admit(b, cases.supersonic_tgv_spec(SIZES[1], precision="fp32_bulk"))[1]  # another group
    print(f"plain {plain} alone {alone} shared {shared} other group {other}", flush=True)
    tuning = min(alone, other) - max(plain)
    assert tuning > 0
    assert max(shared) < max(plain) + 0.5 * tuning


def test_tuned_engines_results_are_the_same():
    specs = _specs()[:2]
    with Batch(hbm_budget=32 << 30, max_cases=4, autotune=True) as b:
        b.tune(specs[1], cases.tgv_state(specs[1]))
        ids = [b.admit(s, None, k) for s, k in zip(specs, (1, 3))]  # together, then the second alone
        while b.run(8)[1]:
            pass
        got = {i: b.retire(i) for i in b.done()}
    for i, s, k in zip(ids, specs, (1, 3)):
        with Solver(s) as alone:
            alone.init_state(s.device_ic())
            alone.step(k)
            np.testing.assert_array_equal(got[i], alone.get_state())
