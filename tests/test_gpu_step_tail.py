"""The all-physical step (use_cfl_dt) forms the pressure gradient's z part,
RHS - grad p, the projection and the constant planes in one launch, and the
stress divergences' z terms in another.  They are the sums that the separate
entry points form, in the same order, so the fields they leave can be had
from one another to the bit: dpdz from p, div_t's planes, u's and v's lid
copy, the wall and lid rows of w.  Grids: the smallest depth, ragged rows, and
two members."""
import numpy as np
import pytest

import lesgo_amd

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
