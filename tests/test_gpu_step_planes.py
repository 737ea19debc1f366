"""What a step does not store or set again each time: the planes of constants
(ghost level, lid, wall padding) of the z derivatives and stresses, set on the
steps that start from physical fields and kept in both buffers of the
exchanged stresses, and the z derivatives, made when they are read.  Level
counts around the chunk of levels that the stress pass marches (8)."""
import numpy as np
import pytest

from oracle import lesgo_oracle as o
from gpu_util import gpu_case, rel_l2, upload_all

pytestmark = pytest.mark.gpu

BOGUS = -1234567890.0


def check_planes(c, nz, nx, dtype):
    b = float(dtype(BOGUS))
    for n in ("dudz", "dvdz", "dwdz", "txx", "txy", "tyy", "txz", "tyz", "tzz"):
        assert np.all(c.download(n)[0] == b), f"{n}: ghost level"
    for n in ("dwdz", "txx", "txy", "tyy", "tzz"):
        assert np.all(c.download(n)[nz] == b), f"{n}: lid"
    for n in ("dudz", "dvdz", "txz", "tyz"):
        assert np.all(c.download(n)[nz] == 0.0), f"{n}: lid"
    for n in ("dudz", "dvdz"):
        assert np.all(c.download(n)[1][:, nx:] == b), f"{n}: wall padding"


@pytest.mark.parametrize("read", ["each step", "at the end"])
@pytest.mark.parametrize("precision,Nz", [("fp64", 3), ("fp64", 7), ("fp64", 8), ("fp64", 9),
                                          ("fp64", 17), ("mixed", 15), ("mixed", 16)])
def test_derivatives_and_planes(precision, Nz, read):
    p = o.Params(16, 16, Nz, dt=1e-5, initu=False, dyn_init=5)
    sp = o.Spectral(p)
    s = o.initial_condition(p, 2)
    tol = 1e-10 if precision == "fp64" else 2e-5
    dtype = np.float64 if precision == "fp64" else np.float32
    with gpu_case(p, precision) as c:
        upload_all(c, s)
        for n in range(1, 8):              # step 5 runs the dynamic model
            o.step(sp, s)
            (c.step if n < 3 else c.step_graph)(1)
            if read == "each step" or n == 7:
                want = o.rmsdiv(p, s)      # from the stored derivatives alone
                got = c.rmsdiv()
                assert abs(got - want) <= tol * max(1.0, want), (got, want)
                for f, lo, hi in (("dudz", 1, p.nz + 1), ("dvdz", 1, p.nz + 1),
                                  ("dwdz", 1, p.nz)):
                    err = rel_l2(c.download(f)[lo:hi, :, :p.nx], s.f[f][lo:hi, :, :p.nx])
                    assert err <= 100 * tol, f"step {n} {f}: {err:.2e}"
                check_planes(c, p.nz, p.nx, dtype)


def test_planes_of_a_member_that_joins():
    """A member copied in after the others' first steps keeps the planes."""
    import lesgo_amd
    cfg = lesgo_amd.Config(16, 16, 9, dt=1e-5, initu=False)
    with lesgo_amd.Case(cfg, members=2) as c:
        c.set_active(1)
        c.seed_state(1, 0.1, member=0)
        c.set_counters(0, 0)
        c.step(3)
        c.copy_member(0, 1)
        c.set_active(2)
        c.step_graph(3)
        for n in ("dudz", "dwdz", "txx", "txz", "tzz", "u", "w"):
            a, b = c.download(n, member=0), c.download(n, member=1)
            assert np.array_equal(a, b), n
        for k, v in ((0, BOGUS), (c.nz, 0.0)):
            assert np.all(c.download("txz", member=1)[k] == v)
