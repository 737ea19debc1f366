"""Timed cases of the LES time step: what a user of this library has it do.

Each case is one pass of a user's program through the public entry points:
a number of time steps and then the read-back of the flow (an output or a
checkpoint interval), or a few of the replaced subroutines called by
themselves.  ``listed()`` holds the cases, ``draw(rng)`` more of the same
ranges, ``prepare``/``run`` set one up and run one pass, ``work`` counts the
bytes and operations it cannot do without and ``exact`` gives the results of
the operator cases in 64-bit numpy.

Launch choices are the library's own (what ``lesgo_amd.run`` and the Fortran
driver use); no tuning table is loaded.
"""
import ctypes
import math

import numpy as np
import torch

import lesgo_amd
from lesgo_amd import _lib

SPINUP = 20          # untimed steps before the first pass; DYN_init of every fresh start
FIELDS = ("u", "v", "w", "p")


def listed():
    return [
        # the smallest grid of the benchmark and of the parity tests: a step is
        # launches and latency
        dict(name="channel32_fp64", kind="step", nx=32, ny=32, Nz=32, precision="fp64",
             steps=100, members=1, disks=False),
        # the serving loop's smallest grid, one job alone
        dict(name="channel64_mixed", kind="step", nx=64, ny=64, Nz=64, precision="mixed",
             steps=100, members=1, disks=False),
        # odd level count, 3-smooth sides with short transforms (72 and 36,
        # 108 and 54 on the dealiasing grid)
        dict(name="ragged72x36x45_fp64", kind="step", nx=72, ny=36, Nz=45, precision="fp64",
             steps=100, members=1, disks=False),
        # a wind farm with the CFL-adaptive time step (lesgo.conf's use_cfl_dt)
        dict(name="cfl96x48x64_mixed", kind="cfl", nx=96, ny=48, Nz=64, precision="mixed",
             steps=50, members=1, disks=True),
        # the benchmark's half channel, the serving loop's largest grid
        dict(name="channel128_mixed", kind="step", nx=128, ny=128, Nz=128, precision="mixed",
             steps=100, members=1, disks=False),
        # a batch of independent half channels, every other one with disks (an
        # ensemble, or one pool of the serving loop)
        dict(name="ensemble16x96_mixed", kind="step", nx=96, ny=96, Nz=64, precision="mixed",
             steps=50, members=16, disks=True),
        # the headline wind farm in both precisions
        dict(name="farm256_mixed", kind="step", nx=256, ny=256, Nz=192, precision="mixed",
             steps=200, members=1, disks=True),
        dict(name="farm256_fp64", kind="step", nx=256, ny=256, Nz=192, precision="fp64",
             steps=100, members=1, disks=True),
        # a host program that keeps the reference's time loop and calls the
        # replaced subroutines one by one
        dict(name="hostloop96x48x64_fp64", kind="hostloop", nx=96, ny=48, Nz=64,
             precision="fp64", steps=20, members=1, disks=False),
        # derivatives, wall model, advection and pressure as single calls on a
        # serving grid
        dict(name="operators128x64x96_fp64", kind="operators", nx=128, ny=64, Nz=96,
             precision="fp64"),
        # tridag_array with the caller's own coefficients, at the wind farm's size
        dict(name="tridag129x256x193", kind="tridag", nx=256, ny=256, Nz=192),
        # the test filter of one host plane: the smallest call
        dict(name="filter64_fp64", kind="filter", nx=64, ny=64, precision="fp64"),
    ]


# sides of the form 2^a 3^b, multiples of 4
SIDES = (16, 24, 32, 36, 48, 64, 72, 96, 108, 128, 144, 192, 216, 256, 288)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("step", "batch", "cfl", "hostloop", "operators", "tridag", "filter"),
                       (10, 3, 3, 2, 2, 2, 1))[0]
    precision = rng.choice(("fp64", "mixed"))
    nx = SIDES[rng.randrange(len(SIDES))]
    ny = rng.choice([s for s in SIDES if nx / 4 <= s <= 2 * nx])
    Nz = _log_int(rng, 10, 192)
    if kind == "filter":
        return dict(kind=kind, nx=nx, ny=ny, precision=precision)
    if kind == "tridag":
        return dict(kind=kind, nx=nx, ny=ny, Nz=Nz)
    if kind == "operators":
        return dict(kind=kind, nx=nx, ny=min(ny, 144), Nz=min(Nz, 96), precision=precision)
    members = 1
    if kind == "batch":
        kind = "step"
        members = max(2, min(rng.randrange(2, 21), int(1.2e7 / (nx * ny * Nz))))
    pts = nx * ny * Nz * members
    if pts > 256 * 256 * 192:
        members = 1
        pts = nx * ny * Nz
        while pts > 256 * 256 * 192:
            Nz = Nz * 3 // 4
            pts = nx * ny * Nz
    cost = pts * (2 if precision == "fp64" else 1) * (2 if kind != "step" else 1)
    steps = 5 * max(2, min(20, int(1.0e9 / cost) // 5))
    disks = rng.random() < 0.5 and nx >= 48 and ny >= 24 and Nz >= 24 and kind != "hostloop"
    return dict(kind=kind, nx=nx, ny=ny, Nz=Nz, precision=precision, steps=steps,
                members=members, disks=disks)


# ---------------------------------------------------------------------------
# Setting a case up
# ---------------------------------------------------------------------------
def _config(case):
    """Fresh start at the benchmark's time steps, the dynamic model from
    step SPINUP on."""
    big = max(case["nx"], case["ny"], case["Nz"]) > 128
    return lesgo_amd.Config(case["nx"], case["ny"], case["Nz"], dt=1e-4 if big else 2e-4,
                            precision=case["precision"], initu=False, dyn_init=SPINUP,
                            use_cfl_dt=case["kind"] == "cfl", cfl=0.1)


def _time_loop(c):
    """One step as a host program that keeps the reference's time loop
    makes it (main.f90:130-344): the replaced subroutines in their order."""
    jt, jt_total = c.counters()
    c.set_counters(jt + 1, jt_total + 1)
    for q in "xyz":
        c.copy_field("RHS" + q, "RHS" + q + "_f")
    c.filt_da("u", "dudx", "dudy")
    c.filt_da("v", "dvdx", "dvdy")
    c.filt_da("w", "dwdx", "dwdy")
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


def _flow_case(case, seed):
    """A running simulation past its start: seeded log-law flow, disks,
    SPINUP steps taken."""
    cfg = _config(case)
    M = case["members"]
    c = lesgo_amd.Case(cfg, members=M)
    rng = np.random.default_rng(seed)
    farm = lesgo_amd.aligned_farm(cfg) if M == 1 else \
        lesgo_amd.aligned_farm(cfg, 2, 2, dia=0.15, hub=0.1)
    for m in range(M):
        if M > 1:
            c.set_member(m, float(10.0 ** rng.uniform(-5.0, -3.0)), float(rng.uniform(0.5, 1.5)))
        c.seed_state(int(rng.integers(1 << 30)), 0.1, member=m)
        if case["disks"] and (M == 1 or m % 2 == 1):
            c.turbines_init(farm, member=m)
    c.set_counters(0, 0)
    if case["kind"] == "hostloop":
        for _ in range(SPINUP):
            _time_loop(c)
    else:
        c.step_graph(SPINUP)
    c.synchronize()
    return c


def _operator_fields(case, seed):
    """Log-law flow with noise on levels 1..nz, and divtz, as float64 arrays
    in the library's layout (rounded to what the case holds)."""
    nx, ny, nz = case["nx"], case["ny"], case["Nz"] + 1
    rng = np.random.default_rng(seed)
    z = (np.arange(1, nz + 1) - 0.5) / (nz - 1)
    prof = np.log(z / 1e-4) / 0.4
    f = {}
    for n in ("u", "v", "w", "divtz"):
        a = np.zeros((nz + 1, ny, nx + 2))
        r = rng.uniform(-0.1, 0.1, (nz, ny, nx)) * prof[:, None, None]
        a[1:, :, :nx] = r + (prof[:, None, None] if n == "u" else 0.0)
        f[n] = a
    f["w"][1] = 0.0
    f["w"][nz] = 0.0
    if case["precision"] == "mixed":
        f = {n: a.astype(np.float32).astype(np.float64) for n, a in f.items()}
    return f


def _tridag_arrays(case, seed):
    """The pressure systems' coefficients scaled by a random factor a row,
    and a random right-hand side."""
    lh, ny, n = case["nx"] // 2 + 1, case["ny"], case["Nz"] + 1
    rng = np.random.default_rng(seed)
    kx = np.arange(lh)[None, :]
    ky = 2.0 * np.minimum(np.arange(ny), ny - np.arange(ny))[:, None]
    h2 = float(n - 1) ** 2
    s = rng.uniform(0.5, 1.5, (n, 1, 1))
    a = np.broadcast_to(s * h2, (n, ny, lh)).copy()
    c = a.copy()
    b = -(s * (kx ** 2 + ky ** 2 + 2.0 * h2 + 1.0))
    b[0], c[0] = -1.0, 1.0
    a[n - 1], b[n - 1] = -1.0, 1.0
    r = rng.standard_normal((n, ny, 2 * lh))
    return a, np.ascontiguousarray(b), c, r


def prepare(case, seed):
    kind = case["kind"]
    if kind == "filter":
        cfg = lesgo_amd.Config(case["nx"], case["ny"], 4, precision=case["precision"])
        plane = np.zeros((case["ny"], case["nx"] + 2))
        plane[:, :case["nx"]] = _filter_plane(case, seed)
        return {"case": case, "c": lesgo_amd.Case(cfg), "plane": plane}
    if kind == "tridag":
        arrs = [torch.from_numpy(x).cuda() for x in _tridag_arrays(case, seed)]
        return {"case": case, "arrs": arrs, "u": torch.zeros_like(arrs[3])}
    if kind == "operators":
        cfg = lesgo_amd.Config(case["nx"], case["ny"], case["Nz"], precision=case["precision"])
        c = lesgo_amd.Case(cfg)
        for n, a in _operator_fields(case, seed).items():
            c.upload(n, a)
        c.synchronize()
        return {"case": case, "c": c}
    return {"case": case, "c": _flow_case(case, seed)}


def _filter_plane(case, seed):
    x = np.random.default_rng(seed).standard_normal((case["ny"], case["nx"]))
    return x.astype(np.float32).astype(np.float64) if case["precision"] == "mixed" else x


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def _read(c, case, name, lo, hi=None, member=0):
    """Levels lo.. of a field in the precision the case holds it in; without
    the padding columns and the ghost level that hold no values of the flow
    (level 0 of the velocity is a sentinel)."""
    a = torch.from_numpy(c.download(name, member=member))[lo:hi, :, :case["nx"]]
    return a.to(torch.float32) if case["precision"] == "mixed" else a


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "filter":
        c = state["c"]
        out = [torch.from_numpy(c.test_filter(state["plane"], w)) for w in (2, 4)]
        return [x.to(torch.float32) if case["precision"] == "mixed" else x for x in out]
    if kind == "tridag":
        p = [ctypes.c_void_p(t.data_ptr()) for t in state["arrs"] + [state["u"]]]
        _lib.check(_lib.lib().lg_tridag_array_device(case["nx"] // 2 + 1, case["ny"],
                                                     case["Nz"] + 1, *p, None), "tridag_array")
        return state["u"]
    c = state["c"]
    if kind == "operators":
        c.filt_da("u", "dudx", "dudy")
        c.filt_da("v", "dvdx", "dvdy")
        c.filt_da("w", "dwdx", "dwdy")
        c.ddz_uv("u", "dudz")
        c.ddz_uv("v", "dvdz")
        c.ddz_w("w", "dwdz")
        c.wallstress()
        c.convec()
        c.press_stag_array()
        nz = case["Nz"] + 1
        out = {n: _read(c, case, n, 1, nz) for n in ("dudx", "dvdy", "RHSx", "RHSy", "RHSz",
                                                     "dpdx", "dpdy")}
        out["p"] = _read(c, case, "p", 0)
        return out
    if kind == "hostloop":
        for _ in range(case["steps"]):
            _time_loop(c)
    else:
        c.step_graph(case["steps"])
    # a lone simulation reads what a domain output holds, a batch each
    # member's velocity
    names = FIELDS if case["members"] == 1 else FIELDS[:3]
    return {f"{n}{m}": _read(c, case, n, 0 if n == "p" else 1, member=m)
            for m in range(case["members"]) for n in names}


# ---------------------------------------------------------------------------
# Compulsory work
# ---------------------------------------------------------------------------
def work(case):
    """Of a step: 31.8 field passes a step in the case's precision (mixed: 4
    of them in FP64; one read and one write of every field between the
    global transposes, with everything local to a plane fused) and the
    transforms' 54.8 planes of nx x ny and 9 of the 3/2 grid a level, and the
    fields read back.  Of the other calls: arrays in once, out once, and
    their transforms."""
    kind, nx, ny = case["kind"], case["nx"], case["ny"]
    l1 = 2.5 * math.log2(nx * ny)
    l2 = 2.25 * 2.5 * math.log2(2.25 * nx * ny)
    if kind == "filter":
        n = nx * ny
        return {"bytes": 4 * 8 * n, "flops": 4 * n * l1}
    if kind == "tridag":
        n = (nx // 2 + 1) * ny * (case["Nz"] + 1)
        return {"bytes": (3 * 8 + 2 * 16) * n, "flops": 13 * n}
    n = nx * ny * case["Nz"]
    s = 8 if case["precision"] == "fp64" else 4
    if kind == "operators":
        # u, v, w and divtz in; six derivatives, three d/dz, RHS, p, grad p out
        return {"bytes": (4 + 9 + 3 + 4) * s * n, "flops": n * (26 * l1 + 9 * l2)}
    n *= case["members"]
    step = 254.4 if s == 8 else 143.2
    outs = 4 if case["members"] == 1 else 3
    return {"bytes": n * (step * case["steps"] + 8 * outs),
            "flops": n * case["steps"] * (54.8 * l1 + 9 * l2)}


# ---------------------------------------------------------------------------
# 64-bit results of the operator cases
# ---------------------------------------------------------------------------
class _Waves:
    """Wavenumbers of the nx x ny plane, Lx = 2 pi, Ly = pi; the Nyquist row
    and column carry none."""

    def __init__(self, nx, ny):
        self.nx, self.ny = nx, ny
        kx = np.arange(nx // 2 + 1, dtype=np.float64)
        ky = np.fft.fftfreq(ny, 1.0 / ny)
        self.keep = np.ones((ny, nx // 2 + 1))
        self.keep[:, -1] = 0.0
        self.keep[ny // 2] = 0.0
        self.kx = kx[None, :] * self.keep
        self.ky = 2.0 * ky[:, None] * self.keep

    def fwd(self, f):
        return np.fft.rfft2(f) * self.keep

    def inv(self, F):
        return np.fft.irfft2(F, s=(self.ny, self.nx))

    def cutoff(self, width):
        dx, dy = 2.0 * math.pi / self.nx, math.pi / self.ny
        kc2 = (math.pi / (width * math.sqrt(dx * dy))) ** 2
        return self.keep * (self.kx ** 2 + self.ky ** 2 < kc2)

    def pad(self, F):
        """The plane's field on the 3/2 grid."""
        nx2, ny2 = 3 * self.nx // 2, 3 * self.ny // 2
        h, q = self.ny // 2, self.nx // 2
        G = np.zeros(F.shape[:-2] + (ny2, nx2 // 2 + 1), complex)
        G[..., :h, :q] = F[..., :h, :q]
        G[..., ny2 - h + 1:, :q] = F[..., h + 1:, :q]
        return np.fft.irfft2(G, s=(ny2, nx2)) * 2.25

    def unpad(self, g):
        ny2, h, q = 3 * self.ny // 2, self.ny // 2, self.nx // 2
        G = np.fft.rfft2(g) / 2.25
        F = np.zeros(G.shape[:-2] + (self.ny, q + 1), complex)
        F[..., :h, :q] = G[..., :h, :q]
        F[..., h + 1:, :q] = G[..., ny2 - h + 1:, :q]
        return F


def _thomas(a, b, c, r):
    """Tridiagonal systems along axis 0: a x[k-1] + b x[k] + c x[k+1] = r."""
    n = b.shape[0]
    x, g = np.empty_like(r), np.empty_like(b)
    x[0] = r[0] / b[0]
    bet = b[0]
    for k in range(1, n):
        g[k] = c[k - 1] / bet
        bet = b[k] - a[k] * g[k]
        x[k] = (r[k] - a[k] * x[k - 1]) / bet
    for k in range(n - 2, -1, -1):
        x[k] -= g[k + 1] * x[k + 1]
    return x


def _exact_operators(case, seed):
    W = _Waves(case["nx"], case["ny"])
    nx, nz = case["nx"], case["Nz"] + 1
    dz = 1.0 / (nz - 1)
    f = _operator_fields(case, seed)
    F = {n: W.fwd(f[n][:, :, :nx]) for n in ("u", "v", "w")}
    u, v, w = (W.inv(F[n]) for n in ("u", "v", "w"))
    # the wall's velocity gradient (equilibrium wall model, z0 = 1e-4)
    g = W.cutoff(2)
    uf, vf = W.inv(F["u"][1] * g), W.inv(F["v"][1] * g)
    ua = np.hypot(uf, vf)
    coef = 0.4 * ua / math.log(0.5 * dz / 1e-4) / (0.5 * dz * 0.4) / ua
    # vorticity on levels 1..nz-1, its x and y components on the w levels
    o1, o2, o3 = (np.zeros((nz + 1,) + F["u"].shape[1:], complex) for _ in range(3))
    for k in range(1, nz):
        if k == 1:
            dvdz, dudz = W.fwd(coef * v[1]), W.fwd(coef * u[1])
            wk = 0.5 * (F["w"][1] + F["w"][2])
        else:
            dvdz, dudz = (F["v"][k] - F["v"][k - 1]) / dz, (F["u"][k] - F["u"][k - 1]) / dz
            wk = F["w"][k]
        o1[k] = 1j * W.ky * wk - dvdz
        o2[k] = dudz - 1j * W.kx * wk
        o3[k] = 1j * W.kx * F["v"][k] - 1j * W.ky * F["u"][k]
    U, V, Wb, O1, O2, O3 = (W.pad(x) for x in (F["u"], F["v"], F["w"], o1, o2, o3))
    out = {n: np.zeros_like(u) for n in ("RHSx", "RHSy", "RHSz")}
    for k in range(1, nz):
        up = 0.5 if k < nz - 1 else 0.0
        dn = 0.5 if k > 1 else 0.0
        cx = -V[k] * O3[k] + up * Wb[k + 1] * O2[k + 1] + dn * Wb[k] * O2[k]
        cy = U[k] * O3[k] - up * Wb[k + 1] * O1[k + 1] - dn * Wb[k] * O1[k]
        out["RHSx"][k] = W.inv(W.unpad(cx))
        out["RHSy"][k] = W.inv(W.unpad(cy))
        if k > 1:
            cz = 0.5 * (-(U[k] + U[k - 1]) * O2[k] + (V[k] + V[k - 1]) * O1[k])
            out["RHSz"][k] = W.inv(W.unpad(cz))
    # pressure: dt = 2e-4 (the configuration's default), AB2 weight 3/2
    sc = 1.0 / 1.5 / 2e-4
    D = W.fwd(f["divtz"][:, :, :nx])
    n = nz + 1
    k2 = W.kx ** 2 + W.ky ** 2
    a = np.full((n,) + k2.shape, dz ** -2)
    b = np.broadcast_to(-(k2 + 2.0 * dz ** -2), a.shape).copy()
    c = a.copy()
    r = np.zeros(a.shape, complex)
    r[1:nz] = sc * (1j * W.kx * F["u"][1:nz] + 1j * W.ky * F["v"][1:nz]
                    + (F["w"][2:nz + 1] - F["w"][1:nz]) / dz)
    b[0], c[0], r[0] = -1.0, 1.0, -dz * D[1]
    a[nz], b[nz], r[nz] = -1.0, 1.0, -dz * D[nz]
    lone = k2 == 0.0          # the Nyquist modes; the mean is integrated upward below
    b[:, lone], a[:, lone], c[:, lone], r[:, lone] = 1.0, 0.0, 0.0, 0.0
    P = _thomas(a, b, c, r)
    P[0, 0, 0] = 0.0
    P[1, 0, 0] = -dz * D[1, 0, 0]
    for k in range(2, n):
        P[k, 0, 0] = P[k - 1, 0, 0] + sc * F["w"][k, 0, 0] * dz
    P = P * W.keep
    S = slice(1, nz)
    return {"dudx": W.inv(1j * W.kx * F["u"][S]), "dvdy": W.inv(1j * W.ky * F["v"][S]),
            "RHSx": out["RHSx"][S], "RHSy": out["RHSy"][S], "RHSz": out["RHSz"][S],
            "dpdx": W.inv(1j * W.kx * P[S]), "dpdy": W.inv(1j * W.ky * P[S]), "p": W.inv(P)}


def exact(case, seed):
    """The operator cases' results; None for whole time steps, whose results
    are those of all their operators in turn."""
    kind, nx = case["kind"], case["nx"]
    if kind == "filter":
        W = _Waves(nx, case["ny"])
        F = W.fwd(_filter_plane(case, seed))
        out = []
        for width in (2, 4):
            p = np.zeros((case["ny"], nx + 2))
            p[:, :nx] = W.inv(F * W.cutoff(width))
            out.append(p)
        return out
    if kind == "tridag":
        a, b, c, r = _tridag_arrays(case, seed)
        rc = r[..., 0::2] + 1j * r[..., 1::2]
        x = _thomas(a, b, c, rc)
        # systems whose rows past the first are left as they were, and the
        # last column, which is not solved
        for jy, jx in ((case["ny"] // 2, slice(None)), (0, slice(0, 1))):
            x[1:, jy, jx] = 0.0
            x[0, jy, jx] = rc[0, jy, jx] / b[0, jy, jx]
        x[:, :, -1] = 0.0
        u = np.empty_like(r)
        u[..., 0::2], u[..., 1::2] = x.real, x.imag
        return u
    if kind == "operators" and nx * case["ny"] * case["Nz"] <= 2_000_000:
        return _exact_operators(case, seed)
    return None
