"""The all-physical step (use_cfl_dt) forms the pressure gradient's z part,
RHS - grad p, the projection and the constant planes in one launch, and the
stress divergences' z terms in another.  Checked to the bit: dpdz from p,
div_t against divstress_uv and divstress_w on the same stresses, the constant
planes, u's and v's lid copy, the wall and lid rows of w.  RHS - grad p and
the projected u, v, w against a host loop over the entry points (rhs_ab2,
press_stag_array, rhs_gradp, project), whose convective term rounds
differently: 1e-10 in FP64, twice the length tests' 2e-5 in mixed (both sides
in float).  Grids: the smallest depth, ragged rows, and two members."""
import numpy as np
import pytest

import lesgo_amd
from lesgo_amd import _lib
from gpu_util import rel_l2

pytestmark = pytest.mark.gpu

BOGUS = -1234567890.0


@pytest.mark.parametrize("nx,ny,Nz,members", [(8, 8, 3, 1), (16, 12, 9, 1), (36, 24, 17, 2)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_physical_step_tail(nx, ny, Nz, members, precision):
    cfg = lesgo_amd.Config(nx, ny, Nz, precision=precision, use_cfl_dt=True, cfl=0.05)
    c = lesgo_amd.Case(cfg, members=members)
    for m in range(members):
        c.seed_state(11 + m, 0.1, member=m)
    c.set_counters(0, 0)
    c.step_graph(3)
    T = np.float64 if precision == "fp64" else np.float32
    bog = float(T(BOGUS))
    nz = Nz + 1
    for m in range(members):
        f = {n: c.download(n, member=m).astype(T) for n in
             ("u", "v", "w", "p", "dpdx", "dpdy", "dpdz", "divtx", "divty", "divtz",
              "RHSx", "RHSy", "RHSz")}
        i = slice(0, nx)
        dz = T(cfg.lz / Nz)
        want = (f["p"][1:nz + 1, :, i] - f["p"][0:nz, :, i]) / dz
        assert np.array_equal(f["dpdz"][1:nz + 1, :, i], want)
        for n in ("u", "v"):
            assert np.array_equal(f[n][nz], f[n][nz - 1])
            assert np.isfinite(f[n][1:nz, :, i]).all()
        for n in ("u", "v", "w", "divtx", "divty", "divtz", "RHSx", "RHSy", "RHSz"):
            assert (f[n][0] == bog).all(), n
        for n in ("dpdx", "dpdy", "divtx", "divty", "RHSx", "RHSy"):
            assert (f[n][nz] == bog).all(), n
        assert (f["w"][1] == 0).all() and (f["w"][nz] == 0).all()
        for n in ("divtx", "divty", "divtz"):
            assert (f[n][1:nz, :, nx:] == 0).all(), n


GRIDS = [(8, 8, 3, 1), (16, 12, 9, 1), (36, 24, 17, 2)]


def started(nx, ny, Nz, members, precision):
    cfg = lesgo_amd.Config(nx, ny, Nz, precision=precision, use_cfl_dt=True, cfl=0.05,
                           initu=False, dyn_init=100)
    c = lesgo_amd.Case(cfg, members=members)
    for m in range(members):
        c.seed_state(11 + m, 0.1, member=m)
    c.set_counters(0, 0)
    return c


@pytest.mark.parametrize("nx,ny,Nz,members", GRIDS)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_divergence_same_bits_as_the_entry_points(nx, ny, Nz, members, precision):
    with started(nx, ny, Nz, members, precision) as c:
        c.step(3)
        names = ("divtx", "divty", "divtz")
        step = {(n, m): c.download(n, member=m) for n in names for m in range(members)}
        zero = np.zeros(c.shape)
        for n, m in step:
            c.upload(n, zero, member=m)
        c.divstress_uv()
        c.divstress_w()
        for (n, m), a in step.items():
            b = c.download(n, member=m)
            assert np.array_equal(a[:Nz + 1], b[:Nz + 1]), (n, m)
            assert np.array_equal(a[Nz + 1, :, :nx], b[Nz + 1, :, :nx]), (n, m)


def host_step(c):
    """One step as a host program makes it (main.f90:130-344)."""
    jt, jt_total = c.counters()
    c.set_counters(jt + 1, jt_total + 1)
    _lib.check(_lib.lib().lg_advance_clock(c._h), "advance_clock")
    for q in "xyz":
        c.copy_field("RHS" + q, "RHS" + q + "_f")
    for f in "uvw":
        c.filt_da(f, f"d{f}dx", f"d{f}dy")
    c.ddz_uv("u", "dudz")
    c.ddz_uv("v", "dvdz")
    c.ddz_w("w", "dwdz")
    c.wallstress()
    c.sgs_stag()
    c.divstress_uv()
    c.divstress_w()
    c.convec()
    c.rhs_ab2()
    c.press_stag_array()
    c.rhs_gradp()
    c.project()


@pytest.mark.parametrize("nx,ny,Nz,members", GRIDS)
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 4e-5)])
def test_tail_against_the_entry_points(nx, ny, Nz, members, precision, tol):
    a = started(nx, ny, Nz, members, precision)
    b = started(nx, ny, Nz, members, precision)
    with a, b:
        a.step(4)
        for _ in range(4):
            host_step(b)
        nz = Nz + 1
        for m in range(members):
            for n, hi in (("u", nz + 1), ("v", nz + 1), ("w", nz + 1), ("RHSx", nz),
                          ("RHSy", nz), ("RHSz", nz), ("dpdx", nz), ("dpdy", nz),
                          ("dpdz", nz + 1), ("p", nz + 1)):
                e = rel_l2(a.download(n, member=m)[1:hi, :, :nx],
                           b.download(n, member=m)[1:hi, :, :nx])
                print(f"  {nx}x{ny}x{Nz} {precision} {n}: {e:.1e}", flush=True)
                assert e <= tol, (n, m, e)
