"""ox_footprint and ox2d_footprint say what a handle allocates: every array of its
one allocation starts at a multiple of 256 bytes.  (No device is needed.)"""
import pytest

from ouxsbli_amd import cases2d
from ouxsbli_amd.batch import footprint
from ouxsbli_amd.cases import CaseSpec

PARTIALS = 4096 * (2 * 5 + 1) * 8  # the diagnostics' sums and compensations of five quantities, and a maximum


def _up(n):
    return (n + 255) // 256 * 256


def _spec(n, prec, visc, rk):
    return CaseSpec(nx=n[0], ny=n[1], nz=n[2], order=4, scheme="KEEP", visc=visc, visc_order=4 if visc != "Euler" else 0,
                    tvd="none", slau_variant="HRSLAU2", rk=rk, precision=prec, threshold=0.4, dt=1e-3, Lx=1.0, Ly=1.0,
                    Lz=1.0)


@pytest.mark.parametrize("rk", [3, 4])
@pytest.mark.parametrize("visc", ["Euler", "NS", "LES"])
@pytest.mark.parametrize("prec", ["fp64", "fp32_bulk"])
@pytest.mark.parametrize("n", [(13, 13, 13), (16, 16, 16), (17, 15, 19)])
def test_footprint_counts_the_padding(n, prec, visc, rk):
    nc, pe = n[0] * n[1] * n[2], 8 if prec == "fp64" else 4
    want = 2 * _up(40 * nc) + _up(5 * nc * pe) + (_up(40 * nc) if rk == 4 else 0)
    want += 2 * (8 if visc == "LES" else 6) * _up(nc * pe) + _up(PARTIALS)
    assert footprint(_spec(n, prec, visc, rk)) == want


@pytest.mark.parametrize("prec", ["fp64", "fp32_bulk"])
def test_footprint_2d_counts_the_padding(prec):
    def f(nx, ny):
        return footprint(cases2d.os_spec(nx=nx, ny=ny, precision=prec))

    tables = f(8, 8) - 3 * 8 * 8 * 32  # 2048 B a state: whole 256 B
    assert 0 < tables < 16384
    for nx, ny in ((9, 9), (257, 129), (31, 33)):
        assert f(nx, ny) == 3 * _up(32 * nx * ny) + tables
