"""The boundary fill's single launch, over every combination of the three kinds.

Ghost primitives and the sensors of the inner ghost layers come from interior
cells alone, also in the edges and corners where directions meet; the states with
their ghost layers and a right-hand side of the result equal the CPU oracle bit
for bit.
"""
import itertools

import numpy as np
import pytest

from ouxsbli_amd.batch import Batch
from ouxsbli_amd.cases import CaseSpec
from ouxsbli_amd.solver import Solver
from oracle_lib import Oracle
from test_bc import _field

pytestmark = pytest.mark.gpu

KINDS = ("periodic", "slip", "extrapolate")
COMBOS = [bc for bc in itertools.product(KINDS, repeat=3) if bc != ("periodic",) * 3]


def _case(bc, order):
    nx, ny, nz = 15, 13, 14
    spec = CaseSpec(nx=nx + order, ny=ny + order, nz=nz + order, order=order, scheme="Hybrid" if order > 2 else "SLAU",
                    visc="Euler", visc_order=0, tvd="hybrid", slau_variant="HRSLAU2", rk=3, precision="fp64",
                    threshold=0.4, dt=1e-3, Lx=1.0, Ly=0.9, Lz=1.1, bc=bc)
    h = order // 2
    Q = np.zeros(spec.state_shape())
    Q[h:-h, h:-h, :, h:-h] = _field((nz, ny, nx), seed=order)
    o = Oracle(spec)
    o.set_qj(Q)
    o.set_bc()
    return spec, o.get_qj()


@pytest.mark.parametrize("order", [2, 6])
@pytest.mark.parametrize("bc", COMBOS, ids="-".join)
def test_bc_fill_bitwise(bc, order):
    spec, Q = _case(bc, order)
    print(f"boundary fill {bc} ORDER {order}", flush=True)
    o = Oracle(spec)
    o.set_state(Q)
    o.step(2)
    with Solver(spec) as s:
        s.set_state(Q)
        s.step(2)
        QJ = s.get_qj()
        Rg = s.rhs()
    h = order // 2
    sl = (slice(h, -h), slice(h, -h), slice(None), slice(h, -h))
    np.testing.assert_array_equal(QJ, o.get_qj())
    np.testing.assert_array_equal(Rg[sl], o.rhs()[sl])


def test_bc_fill_batched_bitwise():
    built = [_case(bc, 6) for bc in COMBOS[::4]]
    with Batch(hbm_budget=4 << 30, max_cases=len(built), autotune=False) as b:
        ids = [b.admit(s, q, 2) for s, q in built]
        b.run(2)
        got = {i: b.retire(i) for i in b.done()}
    for i, (s, q) in zip(ids, built):
        o = Oracle(s)
        o.set_state(q)
        o.step(2)
        np.testing.assert_array_equal(got[i], o.get_state())
