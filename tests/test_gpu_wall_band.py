"""The wall model's test-filtered velocity, taken from the resident spectra's
2-delta band, on grids where the band reaches the last stored column
(kx = nx/2 - 1; in the default domain every grid with ny = 2 nx), for each
column kernel's lengths.  A fresh start against the oracle; tolerances of the
whole-step tests (1e-10) and, mixed, of the length tests (2e-5)."""
import pytest

from oracle import lesgo_oracle as o
from gpu_util import gpu_case, rel_l2, upload_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 2e-5)])
@pytest.mark.parametrize("nx,ny,Nz", [(8, 12, 16), (16, 32, 8), (36, 72, 5), (64, 128, 8)])
def test_wall_stress_where_the_band_is_widest(nx, ny, Nz, precision, tol):
    p = o.Params(nx, ny, Nz, dt=1e-5, initu=False)
    sp = o.Spectral(p)
    s = o.initial_condition(p, 4)
    with gpu_case(p, precision) as c:
        upload_all(c, s)
        for _ in range(3):
            o.step(sp, s)
        c.step(3)
        for n, lo, hi in (("txz", 1, 2), ("tyz", 1, 2), ("dudz", 1, 2), ("u", 1, p.nz),
                          ("v", 1, p.nz), ("w", 1, p.nz)):
            err = rel_l2(c.download(n)[lo:hi, :, :nx], s.f[n][lo:hi, :, :nx])
            print(f"  {nx}x{ny}x{Nz} {n}: {err:.2e}", flush=True)
            assert err <= tol, f"{n}: rel L2 {err:.3e}"
