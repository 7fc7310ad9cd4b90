"""Tile shapes of the SGS viscosity on the GPU.

Workgroups take 32 x 8 columns of the computed cells (all but the outermost
layer, ghost layers included) and walk 8 planes (4 on small grids), with a rim of one cell on
every side; the ghost cells of the viscosity copy the layer next to the opposite
end (set_bc_mut_common, 3D_solver/src/set_bc_common.f90:296-335).  The interiors
below make the computed cells whole tiles and one cell more in each direction;
every right-hand side and state equals the CPU oracle bit for bit.
"""
import numpy as np
import pytest

from ouxsbli_amd.batch import Batch
from ouxsbli_amd.solver import Solver
from oracle_lib import Oracle
from test_gpu_parity import _perturbed_tgv, _spec

pytestmark = pytest.mark.gpu

# at ORDER 6 the computed cells are the interior and 4 more, at ORDER 4 and 2 more
SCHEMES = {
    "hybrid6": (6, "Hybrid", "LES", 6, "hybrid", "HRSLAU2", 4),
    "keep4": (4, "KEEP", "LES", 4, "none", "HRSLAU2", 3),
}
SIZES = [(28, 12, 12), (29, 13, 13), (60, 20, 21), (31, 14, 14), (13, 30, 15), (92, 61, 61)]


@pytest.mark.parametrize("name", list(SCHEMES))
@pytest.mark.parametrize("n", SIZES)
def test_les_shapes_bitwise(name, n):
    spec = _spec(*SCHEMES[name], n=n, Ma=0.5)
    Q = _perturbed_tgv(spec)
    print(f"LES shapes {name} {n}", flush=True)
    o = Oracle(spec)
    o.set_state(Q)
    with Solver(spec) as s:
        s.set_state(Q)
        h = spec.order // 2
        sl = (slice(h, -h), slice(h, -h), slice(None), slice(h, -h))
        np.testing.assert_array_equal(s.rhs()[sl], o.rhs()[sl])
        s.step(2)
        o.step(2)
        np.testing.assert_array_equal(s.get_state(), o.get_state())


def test_les_shapes_batched_bitwise():
    specs = [_spec(*SCHEMES["hybrid6"], n=n, Ma=0.5) for n in SIZES]
    Q = [_perturbed_tgv(s) for s in specs]
    with Batch(hbm_budget=4 << 30, max_cases=len(specs), autotune=False) as b:
        ids = [b.admit(s, q, 2) for s, q in zip(specs, Q)]
        b.run(2)
        got = {i: b.retire(i) for i in b.done()}
    for i, s, q in zip(ids, specs, Q):
        o = Oracle(s)
        o.set_state(q)
        o.step(2)
        np.testing.assert_array_equal(got[i], o.get_state())
