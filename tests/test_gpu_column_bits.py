"""The column pass (csrc/column.hpp) against the separate kernels it stands for
(LESGO_AMD_COLUMN=0: k_spec_ab2, k_tridag, k_spec_project, k_spec_bc) on the
same grid: the same recurrences with the same roundings, so every field is
the same to the bit, through the Euler step, AB2 steps and dynamic-model steps
(whose clips make a last bit's difference visible), with and without disks,
alone and in a batch; and the pressure solve alone.  Each chunk length and
tile width of the plan, and one chunk and part of one."""
import os

import numpy as np
import pytest

import lesgo_amd

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "w", "p", "RHSx", "RHSy", "RHSz", "RHSx_f", "RHSy_f", "RHSz_f", "dpdz",
          "Cs_opt2", "txz")


def pair(cfg, members=1):
    cases = []
    for env in ("0", None):
        if env:
            os.environ["LESGO_AMD_COLUMN"] = env
        try:
            cases.append(lesgo_amd.Case(cfg, members=members))
        finally:
            os.environ.pop("LESGO_AMD_COLUMN", None)
    return cases


def assert_same(a, b, members, what):
    for m in range(members):
        for n in FIELDS:
            x, y = a.download(n, member=m), b.download(n, member=m)
            assert np.isfinite(x).all(), (what, m, n)
            assert np.array_equal(x, y), (what, m, n, float(np.max(np.abs(x - y))))


# (nx, ny, Nz)
GRIDS = {
    "fp64": [(8, 8, 3), (12, 8, 16), (16, 8, 63), (8, 8, 128), (8, 8, 250), (64, 72, 55),
             (64, 64, 100), (64, 64, 192)],
    "mixed": [(8, 8, 3), (16, 8, 31), (8, 8, 48), (8, 8, 96), (8, 8, 224), (8, 8, 390), (8, 8, 410),
              (96, 96, 33), (128, 64, 64), (128, 64, 81), (128, 64, 150)],
}


@pytest.mark.parametrize("precision,nx,ny,Nz",
                         [(p, *g) for p in GRIDS for g in GRIDS[p]])
def test_step_same_bits(precision, nx, ny, Nz):
    # (the tallest grid's explicit diffusion bounds dt: at 1e-5 it diverges)
    cfg = lesgo_amd.Config(nx, ny, Nz, dt=1e-6, precision=precision, initu=False, dyn_init=6)
    a, b = pair(cfg)
    with a, b:
        for c in (a, b):
            c.seed_state(7, 0.02)
        for n in (1, 3, 8):
            for c in (a, b):
                c.step_graph(n)
            assert_same(a, b, 1, a.counters())


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_with_disks_same_bits(precision):
    cfg = lesgo_amd.Config(48, 32, 24, precision=precision, initu=False, dyn_init=6)
    farm = lesgo_amd.aligned_farm(cfg, 2, 2, dia=0.3, hub=0.3, sx_d=7.0, sy_d=5.0)
    a, b = pair(cfg, members=3)
    with a, b:
        for c in (a, b):
            for m in range(3):
                c.seed_state(m, member=m)
            c.turbines_init(farm, member=1)
            c.set_counters(0, 0)
            c.step_graph(4)
            c.seed_state(11, member=2)     # an Euler step beside AB2 steps
            c.step_graph(7)
        assert_same(a, b, 3, "batch")


@pytest.mark.parametrize("precision,nx,ny,Nz",
                         [(p, *g) for p in GRIDS for g in GRIDS[p]])
def test_pressure_alone_same_bits(precision, nx, ny, Nz):
    a, b = pair(lesgo_amd.Config(nx, ny, Nz, precision=precision))
    rng = np.random.default_rng(nx + Nz)
    f = {}
    for n in ("u", "v", "w", "divtz"):
        f[n] = np.zeros(a.shape)
        f[n][1:, :, :nx] = rng.standard_normal((Nz + 1, ny, nx))
    with a, b:
        for c in (a, b):
            for n, x in f.items():
                c.upload(n, x)
            c.press_stag_array()
        for n in ("p", "dpdx", "dpdy", "dpdz"):
            assert np.array_equal(a.download(n), b.download(n)), n
