"""The step's column pass (csrc/column.hpp) at the level counts and plane
sizes where its cut into chunks can go wrong: one chunk and part of one, a
chunk boundary at the lid, the last chunk of a wave and of the block, each
chunk length and tile width its plan uses, plane sizes that do not fill the
last tile, and a grid too tall for it (the separate kernels).  A fresh start
(Euler step, then AB2 steps) against the oracle, and the pressure solve alone
(the same chunked solve, on the physical path).

Tolerances: FP64 as the whole-step tests (1e-10); mixed as the length tests
(inputs and every transform in float, 2e-5)."""
import numpy as np
import pytest

from oracle import lesgo_oracle as o
from gpu_util import gpu_case, rel_l2, upload_all

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-10, "mixed": 2e-5}

# (nx, ny, Nz): nz = Nz + 1 levels
GRIDS = {
    "fp64": [(8, 8, 3), (8, 8, 4), (12, 8, 15), (12, 8, 16), (8, 8, 63), (8, 8, 64), (8, 8, 128),
             (8, 8, 250), (8, 8, 330), (8, 8, 420), (64, 64, 3), (64, 72, 55), (64, 64, 89),
             (64, 64, 100), (64, 64, 192)],
    "mixed": [(8, 8, 3), (12, 8, 7), (16, 8, 31), (8, 8, 48), (8, 8, 71), (8, 8, 72), (8, 8, 96),
              (8, 8, 224), (8, 8, 390), (8, 8, 420), (128, 64, 3), (96, 96, 33), (128, 64, 48),
              (128, 64, 64), (128, 64, 81), (128, 64, 150), (128, 64, 230)],
}
CASES = [(p, *g) for p in GRIDS for g in GRIDS[p]]


def params(nx, ny, Nz, **kw):
    return o.Params(nx, ny, Nz, dt=1e-5, **kw)


@pytest.mark.parametrize("precision,nx,ny,Nz", CASES)
def test_fresh_start_steps(precision, nx, ny, Nz):
    p = params(nx, ny, Nz, initu=False)
    sp = o.Spectral(p)
    s = o.initial_condition(p, 3)
    with gpu_case(p, precision) as c:
        upload_all(c, s)
        for _ in range(3):
            o.step(sp, s)
        c.step(3)
        for n, lo, hi in (("u", 1, p.nz + 1), ("v", 1, p.nz + 1), ("w", 1, p.nz + 1),
                          ("p", 0, p.nz + 1), ("RHSx", 1, p.nz), ("RHSy", 1, p.nz),
                          ("RHSz", 1, p.nz), ("RHSx_f", 1, p.nz), ("RHSz_f", 1, p.nz)):
            err = rel_l2(c.download(n)[lo:hi, :, :nx], s.f[n][lo:hi, :, :nx])
            print(f"  {nx}x{ny}x{Nz} {n}: {err:.2e}", flush=True)
            assert err <= TOL[precision], f"{n}: rel L2 {err:.3e}"


@pytest.mark.parametrize("precision,nx,ny,Nz", CASES)
def test_pressure_alone(precision, nx, ny, Nz):
    p = params(nx, ny, Nz)
    sp = o.Spectral(p)
    s = o.initial_condition(p, 5)
    rng = np.random.default_rng(1)
    s.divtz[1:, :, :nx] = rng.standard_normal((p.nz, ny, nx))
    with gpu_case(p, precision) as c:
        upload_all(c, s)
        c.upload("divtz", s.divtz)
        c.press_stag_array()
        o.press_stag_array(sp, s)
        for n, lo in (("p", 0), ("dpdx", 1), ("dpdy", 1), ("dpdz", 1)):
            err = rel_l2(c.download(n)[lo:p.nz, :, :nx], s.f[n][lo:p.nz, :, :nx])
            print(f"  {nx}x{ny}x{Nz} {n}: {err:.2e}", flush=True)
            assert err <= TOL[precision], f"{n}: rel L2 {err:.3e}"
