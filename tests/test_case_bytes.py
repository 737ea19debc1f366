"""lg_case_bytes, which the serving loop's admission goes by (no GPU calls):
what a case that keeps its spectra between steps holds beyond one that does
not, and the bytes a member may take."""
import ctypes as C

import pytest

import lesgo_amd
from lesgo_amd import _lib


def case_bytes(members, **kw):
    b = C.c_double()
    cfg = lesgo_amd.Config(96, 48, 64, **kw)
    _lib.check(_lib.lib().lg_case_bytes(C.byref(cfg.to_c()), members, C.byref(b)), "case_bytes")
    return b.value


@pytest.mark.parametrize("precision,size", [("fp64", 8), ("mixed", 4)])
@pytest.mark.parametrize("members", [1, 5])
def test_spectral_state(precision, size, members):
    """RHS, RHS_f and the disk forcing (three volumes each) and the pressure
    of two steps; the previous step's disk forcing and vertical stresses."""
    nx, ny, nz = 96, 48, 65
    spectrum = (nz + 1) * ny * (nx // 2) * 2 * size
    field = (nz + 1) * ny * (nx + 2) * size
    kept = case_bytes(members, precision=precision)
    physical = case_bytes(members, precision=precision, use_cfl_dt=True)
    assert kept - physical == members * (11 * spectrum + 6 * field)


@pytest.mark.parametrize("precision,one,two", [("fp64", 398317688, 795373808),
                                               ("mixed", 205804664, 410366192)])
def test_budget_holds_what_it_held(precision, one, two):
    """One and two members fit the bytes they took when the step's AB2,
    pressure solve and projection were separate kernels."""
    assert case_bytes(1, precision=precision) <= one
    assert case_bytes(2, precision=precision) <= two
