"""What a program does with this package, as timed cases.

listed() names them, draw() gives others of the same ranges, prepare() makes
what a program has in hand before the call (handle, fields, particles, right-
hand sides), run() is one pass through the public entry points, work() what a
pass cannot do without, and exact() the same results from plain torch and
numpy in 64 bits.

Four kinds of work, as the drivers, the benchmark and the tests use them:

  step       RK3 steps of one ring on its handle; the fields stay in device
             memory and are read there (vrh_device_ptr).  With particles: steps,
             then the download of the particles, as an export does.
  ensemble   one RK3 step of several rings by one graph launch.
  poisson    the standalone pressure solve, host arrays in and out.
  helmholtz  the per-mode (r, z) systems on the tanh grid, host arrays in and
             out, by the direct solve or by conjugate gradients.
"""
import math
import random

import numpy as np
import torch

import vring_amd

RMAX, ZMAX = 4.0, 12.0
DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64


def _step(nt, nr, nz, precision, Re, **more):
    return dict(dict(kind="step", nt=nt, nr=nr, nz=nz, precision=precision, Re=Re, rings=1, mesh="uniform", steps=1,
                     particles="none", np=0), **more)


def listed():
    return [
        # the smallest ring of the benchmark's parity workload: a step of a
        # few hundred thousand cells, latency and launches
        dict(_step(32, 64, 128, "fp64", 1000.0), name="step_small"),
        # the grid of the reference's VR3Dlight deck: an odd number of theta
        # points, as the reference's transforms want it
        dict(_step(129, 128, 128, "fp64", 500.0), name="step_deck_odd"),
        # no length a power of two (the grid of the analysis tests), mixed precision
        dict(_step(33, 96, 200, "mixed", 1000.0), name="step_ragged_mixed"),
        # the headline ring in both precisions
        dict(_step(128, 256, 512, "mixed", 3000.0), name="step_headline_mixed"),
        dict(_step(128, 256, 512, "fp64", 3000.0), name="step_headline"),
        # the large workload's grid with its two rings
        dict(_step(256, 512, 1024, "mixed", 7500.0, rings=2, rmax=5.0, zmax=20.0), name="step_large_mixed"),
        # axial points gathered at the inlet: dense z transforms
        dict(_step(64, 128, 256, "fp64", 3000.0, mesh="tanh"), name="step_stretched"),
        # tracers carried and exported: trilinear RK3, a million of them
        dict(_step(64, 128, 256, "mixed", 2000.0, steps=2, particles="trilinear_rk3", np=1000000),
             name="particles_trilinear"),
        # the reference's particle scheme with its five sub-steps, one batch
        # of an ensemble ring's size
        dict(_step(64, 96, 256, "fp64", 2000.0, steps=1, particles="lsq_euler", np=50000), name="particles_lsq"),
        # eight rings of the ensemble workload's shapes
        dict(kind="ensemble", members=8, shapes=3, name="ensemble"),
        # a caller's own right-hand side
        dict(kind="poisson", nt=64, nr=128, nz=256, precision="fp64", theta="consistent", name="poisson"),
        # 64 azimuthal modes of the stretched-grid pressure operator
        dict(kind="helmholtz", nr=256, nz=512, slots=64, method="pcg", tol=1e-8, name="helmholtz_pcg"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    u = rng.random()
    if u < 0.62:
        precision = rng.choice(["fp64", "mixed"])
        Re = round(math.exp(rng.uniform(math.log(500.0), math.log(7500.0))), 1)
        v = rng.random()
        if v < 0.35:  # power-of-two transforms, any number of radial rows
            nt, nz = rng.choice([32, 64, 128, 256]), rng.choice([64, 128, 256, 512])
            return _step(nt, _logint(rng, 48, 300), nz, precision, Re)
        if v < 0.6:  # any lengths
            while True:
                nt, nr, nz = _logint(rng, 9, 200), _logint(rng, 32, 200), _logint(rng, 48, 420)
                if nt * nr * nz * nz <= 600000000:
                    return _step(nt, nr, nz, precision, Re)
        if v < 0.75:
            return _step(rng.choice([32, 64, 128]), _logint(rng, 48, 200), _logint(rng, 64, 300), precision, Re,
                         mesh="tanh")
        nt, nr, nz = rng.choice([32, 64, 128]), _logint(rng, 64, 160), rng.choice([128, 256])
        if rng.random() < 0.6:
            return _step(nt, nr, nz, precision, Re, steps=rng.choice([1, 2, 5]), particles="trilinear_rk3",
                         np=_logint(rng, 20000, 1000000))
        return _step(nt, nr, nz, precision, Re, particles="lsq_euler", np=_logint(rng, 2000, 60000))
    if u < 0.72:
        return dict(kind="ensemble", members=rng.randint(2, 8), shapes=rng.randrange(1000))
    if u < 0.86:
        pow2 = rng.random() < 0.6
        return dict(kind="poisson", nt=rng.choice([16, 32, 64, 128]) if pow2 else _logint(rng, 9, 150),
                    nr=_logint(rng, 24, 200), nz=rng.choice([64, 128, 256]) if pow2 else _logint(rng, 40, 300),
                    precision=rng.choice(["fp64", "mixed"]), theta=rng.choice(["consistent", "exact_m2"]))
    return dict(kind="helmholtz", nr=16 * rng.randint(4, 16), nz=_logint(rng, 64, 512), slots=rng.randint(4, 64),
                method=rng.choice(["pcg", "direct"]), tol=1e-8)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
class _Grid:
    """Sizes and meshes of a case, arrays over j = 0..nr+2 and k = 0..nz+2."""

    def __init__(self, nt, nr, nz, rmax=RMAX, zmax=ZMAX, stretch=0.0):
        self.nt, self.nr, self.nz, self.rmax, self.zmax, self.stretch = nt, nr, nz, rmax, zmax, stretch
        self.dth, self.dr, self.dz = 2.0 * math.pi / nt, rmax / nr, zmax / nz
        j = np.arange(nr + 3)
        self.rm, self.rc = (j - 0.5) * self.dr, (j - 1.0) * self.dr
        zf = np.arange(nz + 1) * self.dz  # faces z(1)..z(nz+1)
        if stretch:
            zf = zmax * (1.0 + np.tanh(stretch * (np.arange(nz + 1) / nz - 1.0)) / np.tanh(stretch))
            zf[0], zf[-1] = 0.0, zmax
        self.zf = zf
        # what vrh_set_axial_mesh takes, k = 0..nz+1: centres, faces, dz/dzeta
        zm = np.zeros(nz + 2)
        zm[1:-1] = 0.5 * (zf[1:] + zf[:-1])
        zm[0], zm[-1] = -zm[1], 2.0 * zmax - zm[nz]
        dmz, dcz = np.zeros(nz + 2), np.zeros(nz + 2)
        dmz[1:-1] = (zf[1:] - zf[:-1]) / self.dz
        dmz[0], dmz[-1] = dmz[1], dmz[nz]
        dcz[1:] = (zm[1:] - zm[:-1]) / self.dz
        dcz[0] = dcz[1]
        self.axial = zm, np.concatenate([[-zf[1]], zf]), dmz, dcz

    def shape(self):  # a haloed field, theta fastest
        return self.nz + 3, self.nr + 3, self.nt


def _agm_ke(k1):
    """Complete elliptic integrals K, E of the complementary modulus k1."""
    a, b = torch.ones_like(k1), k1.clone()
    s, w = 1.0 - k1 * k1, 1.0
    s = 1.0 - 0.5 * s
    for _ in range(6):
        c = 0.5 * (a - b)
        a, b = 0.5 * (a + b), torch.sqrt(a * b)
        s = s - w * c * c
        w *= 2.0
    K = 0.5 * math.pi / a
    return K, K * s


def _ring_fields(g, rings, amp, phases):
    """Haloed q1, q2, q3 of smoothed ring filaments (R, z0, sigma, Gamma) whose
    radius is R + amp sum_m cos(m theta + phase), m = 2, 3, ...: their Stokes
    streamfunction, tapered to zero at the inlet and the wall, differenced
    on the staggered grid, so that the field is discretely solenoidal."""
    dev = DEV
    rc = torch.tensor(g.rc[1:g.nr + 2], dtype=F64, device=dev)[None, :, None]
    zf = torch.tensor(g.zf, dtype=F64, device=dev)[:, None, None]
    th = (torch.arange(g.nt, dtype=F64, device=dev) + 0.5) * g.dth
    dR = sum(amp * torch.cos((m + 2) * th + p) for m, p in enumerate(phases))[None, None, :]
    taper = (1.0 - (rc / g.rmax) ** 2) ** 2 * (1.0 - torch.exp(-zf * zf)) * (1.0 - torch.exp(-(g.zmax - zf) ** 2))
    psi = torch.zeros(g.nz + 1, g.nr + 1, g.nt, dtype=F64, device=dev)
    for R, z0, sigma, gam in rings:
        d2 = (zf - z0) ** 2 + sigma * sigma
        p1, p2 = torch.sqrt(d2 + (rc - R - dR) ** 2), torch.sqrt(d2 + (rc + R + dR) ** 2)
        lam = (p2 - p1) / (p2 + p1)
        K, E = _agm_ke(torch.sqrt(1.0 - lam * lam))
        psi += gam / (2.0 * math.pi) * (p1 + p2) * (K - E) * taper
        del d2, p1, p2, lam, K, E
    q = [torch.zeros(g.shape(), dtype=F64, device=dev) for _ in range(3)]
    dz = torch.tensor(np.diff(g.zf), dtype=F64, device=dev)[:, None, None]
    rm = torch.tensor(g.rm[1:g.nr + 1], dtype=F64, device=dev)[None, :, None]
    q[1][1:g.nz + 1, 2:g.nr + 1] = -((psi[1:] - psi[:-1]) / dz)[:, 1:g.nr]
    q[2][1:g.nz + 1, 1:g.nr + 1] = ((psi[:, 1:] - psi[:, :-1]) / (g.dr * rm))[:-1]
    return q


def _cfl_dt(g, q, cfl=0.3, jet=1.0):
    dev = q[0].device
    rc = torch.tensor(g.rc[2:g.nr + 1], dtype=F64, device=dev)[None, :, None]
    dz = torch.tensor(np.diff(g.zf), dtype=F64, device=dev)[:, None, None]
    u = q[2][1:g.nz + 1, 1:g.nr + 1].abs() / dz
    u[:, 1:] += (q[1][1:g.nz + 1, 2:g.nr + 1] / rc).abs() / g.dr
    return cfl / max(float(u.max()), jet / float(np.diff(g.zf).min()))


def _flow(case, seed):
    """Grid, initial fields and time step of a ring, from the seed alone."""
    r = np.random.Generator(np.random.PCG64(seed))
    g = _Grid(case["nt"], case["nr"], case["nz"], case.get("rmax", RMAX), case.get("zmax", ZMAX),
              2.0 if case.get("mesh") == "tanh" else 0.0)
    core = case.get("sigma", 0.2)
    z0 = float(r.uniform(2.5, 3.5))
    rings = [(float(r.uniform(0.9, 1.1)), z0 + 1.0 * n, core * float(r.uniform(0.9, 1.1)), float(r.uniform(0.8, 1.2)))
             for n in range(case.get("rings", 1))]
    q = _ring_fields(g, rings, 0.02, r.uniform(0.0, 2.0 * math.pi, 7))
    return g, q, _cfl_dt(g, q), rings


def _particles(case, seed, rings):
    """Rows (x, y, z, velocity, ...) uniform in the torus around the ring's core."""
    r = np.random.Generator(np.random.PCG64(seed + 77))
    n = case["np"]
    R, z0 = rings[0][0], rings[0][1]
    a = 0.6 * np.sqrt(r.random(n))
    phi, th = 2.0 * math.pi * r.random(n), 2.0 * math.pi * r.random(n)
    rad = R + a * np.cos(phi)
    u = np.zeros((n, 6 if case["particles"] == "trilinear_rk3" else 117))
    u[:, 0], u[:, 1], u[:, 2] = rad * np.cos(th), rad * np.sin(th), z0 + a * np.sin(phi)
    if u.shape[1] == 117:
        u[:, [6, 10, 14]] = 1.0
    return u


_NSUB = 5  # the reference's sub-steps of a particle batch


class _Mem:
    """A device array of a solver, kept alive with its solver."""

    def __init__(self, solver, name, shape):
        self.solver = solver
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "version": 3,
                                         "data": (solver.device_ptr(name), False)}


_FIELDS = ("q1", "q2", "q3", "pres")


def _solver(case, seed):
    g, q, dt, rings = _flow(case, seed)
    s = vring_amd.Solver(g.nt, g.nr, g.nz, g.rmax, g.zmax, case["Re"], dt, precision=case["precision"])
    if g.stretch:
        s.set_axial_mesh(*g.axial)
    fields = {n: torch.as_tensor(_Mem(s, n, g.shape()), device="cuda") for n in _FIELDS}
    for n, a in zip(_FIELDS, q):
        fields[n].copy_(a)
    if case.get("particles", "none") != "none":
        s.particles_create([case["np"]], [vring_amd.lib.stokes_number(5.0e-6 / 0.02, case["Re"])], [_NSUB],
                           case["particles"])
        s.particles_upload(0, _particles(case, seed, rings))
    torch.cuda.synchronize()
    return s, fields


def _members(case):
    """The ensemble workload's shapes and parameters, drawn from the case's own numbers."""
    r = random.Random(case["shapes"])
    return [dict(_step(r.choice([32, 64, 128]), r.choice([64, 96, 128, 192]), r.choice([128, 256, 512]), "mixed",
                       r.uniform(500.0, 5000.0)), sigma=r.uniform(0.1, 0.3)) for _ in range(case["members"])]


def _poisson_rhs(case, seed):
    """A smooth right-hand side with a broad spectrum and zero mean flux, theta fastest: (nz, nr, nt)."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    f = torch.randn(case["nz"], case["nr"], case["nt"], dtype=F64, device=DEV, generator=gen)
    rm = torch.tensor((np.arange(case["nr"]) + 0.5) * RMAX / case["nr"], dtype=F64, device=DEV)[None, :, None]
    return f - (f * rm).sum() / (rm.sum() * case["nt"] * case["nz"])


def _helmholtz_rhs(case, seed):
    """Four Gaussian ring cores per slot, (slots, nz, nr) on the host."""
    r = np.random.Generator(np.random.PCG64(seed))
    g = _Grid(3, case["nr"], case["nz"], stretch=2.0)
    rm = torch.tensor(g.rm[1:g.nr + 1], dtype=F64, device=DEV)
    zm = torch.tensor(0.5 * (g.zf[1:] + g.zf[:-1]), dtype=F64, device=DEV)
    p = torch.tensor(r.random((4, 4, case["slots"])), dtype=F64, device=DEV)[..., None]
    f = torch.zeros(case["slots"], g.nz, g.nr, dtype=F64, device=DEV)
    for c in p:
        s = 0.1 + 0.2 * c[2]
        er = torch.exp(-(((rm - (0.05 + 0.85 * c[0]) * RMAX) / s) ** 2))
        ez = torch.exp(-(((zm - (0.05 + 0.9 * c[1]) * ZMAX) / s) ** 2))
        f += (2.0 * c[3] - 1.0)[..., None] * ez[:, :, None] * er[:, None, :]
    return f.cpu().numpy()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        s, fields = _solver(case, seed)
        return dict(case=case, solver=s, fields=fields)
    if kind == "ensemble":
        made = [_solver(m, seed * 1000 + n) for n, m in enumerate(_members(case))]
        return dict(case=case, ens=vring_amd.Ensemble([s for s, _ in made]), fields=[f for _, f in made])
    if kind == "poisson":
        s = vring_amd.Solver(case["nt"], case["nr"], case["nz"], RMAX, ZMAX, 1000.0, 0.01, theta_eigen=case["theta"],
                             precision=case["precision"])
        rhs = _poisson_rhs(case, seed).cpu().numpy()
        return dict(case=case, solver=s, rhs=rhs.T)  # (nt, nr, nz), Fortran order
    pool = 8 if case["nr"] % 128 == 0 and case["nz"] % 8 == 0 else 1
    hz = vring_amd.Helmholtz(case["nr"], case["nz"], case["slots"], RMAX, ZMAX, 2.0, pool=pool)
    hz.set_modes(np.arange(case["slots"], dtype=np.int32))
    return dict(case=case, hz=hz, f=_helmholtz_rhs(case, seed))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        s = state["solver"]
        s.step(case["steps"])
        if case["np"]:
            u, alive = s.particles_download(0, case["np"])
            return dict(state["fields"], u=u, alive=alive)
        return state["fields"]
    if kind == "ensemble":
        state["ens"].step(1)
        return state["fields"]
    if kind == "poisson":
        return state["solver"].poisson(state["rhs"])
    if case["method"] == "direct":
        return state["hz"].direct(state["f"])
    p, iters, relres, _ = state["hz"].solve(state["f"], case["method"], case["tol"], 5000)
    return dict(p=p, iters=iters)


def work(case):
    kind = case["kind"]
    if kind == "step":
        n = case["nt"] * case["nr"] * case["nz"]
        # a step reads and writes q1..q3, p and the pressure gradient; about
        # 400 operations per cell and substep beside the transforms
        tr = 5.0 * (math.log2(case["nt"]) + math.log2(case["nz"])) if case["mesh"] == "uniform" else \
            5.0 * math.log2(case["nt"]) + 4.0 * case["nz"]
        rows = {"none": 0, "trilinear_rk3": 6, "lsq_euler": 117}[case["particles"]]
        per = {"none": 0.0, "trilinear_rk3": 3 * 150.0, "lsq_euler": _NSUB * 4000.0}[case["particles"]]
        return dict(bytes=112.0 * n + 16.0 * rows * case["np"],
                    flops=case["steps"] * (3.0 * n * (400.0 + tr) + per * case["np"]))
    if kind == "ensemble":
        w = [work(m) for m in _members(case)]
        return dict(bytes=sum(x["bytes"] for x in w), flops=sum(x["flops"] for x in w))
    if kind == "poisson":
        n = case["nt"] * case["nr"] * case["nz"]
        return dict(bytes=16.0 * n, flops=n * (10.0 + 5.0 * (math.log2(case["nt"]) + math.log2(case["nz"]))))
    n = case["nr"] * case["nz"] * case["slots"]
    return dict(bytes=16.0 * n, flops=n * (4.0 * case["nz"] + 10.0))  # the direct solve's


# --------------------------------------------------------------------------
# the same results from plain torch and numpy in 64 bits
# --------------------------------------------------------------------------
def _solve_radial(aa, bb, cc, f):
    """Tridiagonal solve along dim 1 of f (nz, nr, modes): aa, cc (nr), bb like f, real."""
    nr = f.shape[1]
    x = torch.empty_like(f)
    beta = torch.empty_like(bb)
    beta[:, 0] = bb[:, 0]
    x[:, 0] = f[:, 0] / beta[:, 0]
    for j in range(1, nr):
        beta[:, j] = bb[:, j] - aa[j] * cc[j - 1] / beta[:, j - 1]
        x[:, j] = (f[:, j] - aa[j] * x[:, j - 1]) / beta[:, j]
    for j in range(nr - 2, -1, -1):
        x[:, j] -= (cc[j] / beta[:, j]) * x[:, j + 1]
    return x


class _Poisson:
    """The pressure solve of a grid: z eigenvectors (cosines on the uniform
    mesh), theta transform, radial systems; the (0, 0) system is pinned at the wall."""

    def __init__(self, g, theta, dev):
        self.g, self.dev = g, dev
        nz, nr = g.nz, g.nr
        if g.stretch:
            m3, c3 = (1.0 / g.dz) / g.axial[2], (1.0 / g.dz) / g.axial[3]
            d = np.array([m3[k] * ((c3[k] if k > 1 else 0.0) + (c3[k + 1] if k < nz else 0.0))
                          for k in range(1, nz + 1)])
            e = np.array([-math.sqrt(m3[k] * m3[k + 1]) * c3[k + 1] for k in range(1, nz)])
            lam, W = np.linalg.eigh(np.diag(d) + np.diag(e, 1) + np.diag(e, -1))
            lam[0] = 0.0
            sq = np.sqrt(m3[1:nz + 1])
            fwd, inv = W.T / sq[None, :], W * sq[:, None]
        else:
            k = np.arange(nz)
            C = np.cos(math.pi * np.outer(k, k + 0.5) / nz)
            fwd, inv = C / nz, 2.0 * C.T
            inv[:, 0] = 1.0
            lam = 2.0 / g.dz ** 2 * (1.0 - np.cos(math.pi * k / nz))
        self.fwd, self.inv = (torch.tensor(a, dtype=F64, device=dev) for a in (fwd, inv))
        rm = g.rm[1:nr + 1]
        aa, cc = -1.0 / g.dr ** 2 + 0.5 / (rm * g.dr), -1.0 / g.dr ** 2 - 0.5 / (rm * g.dr)
        m = np.arange(g.nt // 2 + 1)
        wth = m.astype(float) ** 2 if theta == "exact_m2" else 2.0 / g.dth ** 2 * (1.0 - np.cos(m * g.dth))
        t = lambda a: torch.tensor(a, dtype=F64, device=dev)  # noqa: E731
        bb = 2.0 / g.dr ** 2 + t(wth)[None, None, :] / t(rm * rm)[None, :, None] + t(lam)[:, None, None]
        bb[:, 0] += aa[0]
        pin = torch.ones(nz, m.size, dtype=F64, device=dev)
        pin[0, 0] = -1.0
        bb[:, nr - 1] += cc[nr - 1] * pin
        aa[0], cc[nr - 1] = 0.0, 0.0
        self.aa, self.bb, self.cc = [float(a) for a in aa], bb, [float(a) for a in cc]

    def __call__(self, rhs):  # (nz, nr, nt)
        nz, nr, nt = rhs.shape
        s = torch.view_as_real(torch.fft.rfft(rhs, dim=2))
        s = (self.fwd @ s.reshape(nz, -1)).reshape(nz, nr, -1, 2)
        s = torch.stack([_solve_radial(self.aa, self.bb, self.cc, s[..., c]) for c in (0, 1)], dim=-1)
        s = (self.inv @ s.reshape(nz, -1)).reshape(nz, nr, -1, 2)
        return torch.fft.irfft(torch.view_as_complex(s.contiguous()), n=nt, dim=2)


def _profile(t):
    t1, u = float(np.float32(0.1)) * 2.0, 0.0
    ramp = lambda x: 3.0 * x * x - 2.0 * x ** 3  # noqa: E731
    if 0.0 < t < t1:
        u = ramp(t / t1)
    if t1 < t < 2.0:
        u = 1.0
    if 2.0 < t < 2.0 + t1:
        u = ramp((2.0 + t1 - t) / t1)
    return u


class _Stepper:
    """The fractional-step RK3 of the flow on one grid, fields (nz+3, nr+3, nt)."""

    RK = {1: (8.0 / 15.0, 0.0), 2: (5.0 / 12.0, -17.0 / 60.0), 3: (3.0 / 4.0, -5.0 / 12.0)}

    def __init__(self, g, Re, dt, q, dev):
        self.g, self.Re, self.dt, self.dev, self.t = g, Re, dt, dev, 0.0
        nr, nz = g.nr, g.nz
        self.poisson = _Poisson(g, "exact_m2", dev)
        z = lambda: torch.zeros(g.shape(), dtype=F64, device=dev)  # noqa: E731
        self.q = [a.to(dev).clone() for a in q]
        self.pres = z()
        self.prg, self.ru = [z() for _ in range(3)], [z() for _ in range(3)]
        self.csort, self.dq3no = (torch.zeros(nr + 3, g.nt, dtype=F64, device=dev) for _ in range(2))
        self.dx = 1.0 / g.dth, 1.0 / g.dr, 1.0 / g.dz
        dx1, dx2, dx3 = self.dx
        rm, rc = g.rm, g.rc
        v = {n: np.zeros(nr + 3) for n in ("h1", "h12", "h1n", "h1a", "h2", "h2p", "h2m", "h2a", "s1", "s1n", "s1s",
                                           "s1c", "s2", "s2p", "s2m", "s3n", "s3s")}
        j = np.arange(1, nr + 1)
        v["h1"][j], v["h12"][j] = 0.25 * dx1 / rm[j], 0.25 * dx2 / rm[j]
        v["h1n"][j], v["h1a"][j] = 0.125 / rm[j] ** 2, dx1 / (Re * rm[j] ** 3)
        v["s1"][j] = (dx1 / rm[j]) ** 2
        v["s1n"][j], v["s1s"][j], v["s1c"][j] = rc[j + 1] ** 3, rc[j] ** 3, (dx2 / rm[j]) ** 2
        v["s3n"][j], v["s3s"][j] = dx2 ** 2 * rc[j + 1] / rm[j], dx2 ** 2 * rc[j] / rm[j]
        i = np.arange(2, nr + 1)
        v["h2"][i], v["h2a"][i], v["s2"][i] = 0.25 * dx1 / rc[i], dx1 / (Re * rc[i]), (dx1 / rc[i]) ** 2
        v["h2p"][i], v["h2m"][i] = 0.25 * dx2 / rm[i], 0.25 * dx2 / rm[i - 1]
        v["s2p"][i], v["s2m"][i] = dx2 ** 2 * rc[i] / rm[i], dx2 ** 2 * rc[i] / rm[i - 1]
        self.v = v
        # z differences at centres (m3) and faces (c3), k = 0..nz+1
        if g.stretch:
            self.m3, self.c3 = dx3 / g.axial[2], dx3 / g.axial[3]
        else:
            self.m3 = self.c3 = np.full(nz + 2, dx3)
        h1, h2 = 0.5 / self.m3[1], 1.0 / self.c3[2]
        self.ws, self.w2 = 2.0 / (h1 * (h1 + h2)), 2.0 / (h2 * (h1 + h2))
        self.da = rm[:nr + 1] / (dx1 * dx2)
        self.qc = np.zeros(nr + 3)
        self.qc[1:nr + 1] = 1.0 - (rm[1:nr + 1] / g.rmax) ** 2
        self.inlet = rc[:nr + 2] <= float(np.float32(0.4999))

    def row(self, name):  # a radial vector over j = 1..nr, broadcast over (k, j, i)
        return torch.tensor(self.v[name][1:self.g.nr + 1], dtype=F64, device=self.dev)[None, :, None]

    def col(self, a, k0, k1):  # an axial vector over k = k0..k1
        return torch.tensor(np.asarray(a)[k0:k1 + 1], dtype=F64, device=self.dev)[:, None, None]

    def _inverse(self, a, b, c, dim):
        n = len(b)
        T = np.diag(np.asarray(b, float)) + np.diag(np.asarray(a[1:], float), -1) + np.diag(np.asarray(c[:-1], float), 1)
        Ti = torch.linalg.inv(torch.tensor(T, dtype=F64, device=self.dev))

        def solve(x):
            if dim == 0:
                return (Ti @ x.reshape(n, -1)).reshape(x.shape)
            return torch.matmul(Ti, x)
        return solve

    def substep(self, irk, t):
        g, dt, Re, v = self.g, self.dt, self.Re, self.v
        nr, nz, nt = g.nr, g.nz, g.nt
        dx1, dx2, dx3 = self.dx
        ga, ro = self.RK[irk]
        al = ga + ro
        R, rm, rc = self.row, g.rm, g.rc
        m3, c3 = self.col(self.m3, 1, nz), self.col(self.c3, 1, nz)
        k, j = slice(1, nz + 1), slice(1, nr + 1)
        ip = lambda a: torch.roll(a, -1, 2)  # noqa: E731
        im = lambda a: torch.roll(a, 1, 2)  # noqa: E731
        up = lambda q: q[2:nz + 2, j]  # noqa: E731
        dn = lambda q: q[0:nz, j]  # noqa: E731
        no = lambda q: q[k, 2:nr + 2]  # noqa: E731
        so = lambda q: q[k, 0:nr]  # noqa: E731

        def jm(q):  # j - 1, the first row its own neighbour
            return torch.cat([q[k, 1:2], q[k, 1:nr]], dim=1)

        q1, q2, q3 = self.q
        a, b, c = q1[k, j], q2[k, j], q3[k, j]
        first = torch.zeros(nz, 1, 1, dtype=torch.bool, device=self.dev)
        first[0] = True
        nil = torch.zeros((), dtype=F64, device=self.dev)
        cm, cp = m3 * c3, m3 * self.col(self.c3, 2, nz + 1)

        def d33c(q, x):
            return torch.where(first, (up(q) - x) * self.w2 - x * self.ws, (up(q) - x) * cp - (x - dn(q)) * cm)

        # ---- explicit terms ----
        n2 = no(q2)
        h = ((ip(a) + a) ** 2 - (im(a) + a) ** 2) * R("h1")
        h = h + ((n2 + im(n2)) * (no(q1) + a) - (a + jm(q1)) * (b + im(b))) * R("h12")
        h = h + ((ip(a) + a) * (n2 + b) + (a + im(a)) * (im(n2) + im(b))) * R("h1n")
        u3 = up(q3)
        h = h + (0.25 * (u3 + im(u3)) * (up(q1) + a) - torch.where(first, nil, 0.25 * (c + im(c)) * (a + dn(q1)))) * m3
        H1 = ((n2 + b) - (im(n2) + im(b))) * R("h1a") - h
        rmt = torch.tensor(rm, dtype=F64, device=self.dev)
        irm = 1.0 / rmt[None, 1:nr + 1, None]
        irn = 1.0 / rmt[None, 2:nr + 2, None]
        irs = 1.0 / torch.cat([rmt[1:2], rmt[1:nr]])[None, :, None]
        D1 = (ip(a) - 2.0 * a + im(a)) * R("s1") + d33c(q1, a) + \
            ((no(q1) * irn - a * irm) * R("s1n") - (a * irm - jm(q1) * irs) * R("s1s")) * R("s1c")

        s1, s2, s3 = so(q1), so(q2), so(q3)
        h = ((ip(a) + ip(s1)) * (ip(b) + b) - (a + s1) * (b + im(b))) * R("h2")
        h = h + (n2 + b) ** 2 * R("h2p") - (b + s2) ** 2 * R("h2m")
        w = 0.5 * (a + ip(a)) + 0.5 * (s1 + ip(s1))
        u3s = q3[2:nz + 2, 0:nr]
        h = h + (0.25 * (u3 + u3s) * (up(q2) + b) - torch.where(first, nil, 0.25 * (c + s3) * (b + dn(q2)))) * m3
        H2 = -((ip(a) + ip(s1)) - (a + s1)) * R("h2a") - (h - 0.25 * w * w)
        D2 = (ip(b) - 2.0 * b + im(b)) * R("s2") + d33c(q2, b) + n2 * R("s2p") - b * (R("s2p") + R("s2m")) + s2 * R("s2m")

        h = ((no(q3) + c) * (n2 + q2[0:nz, 2:nr + 2]) - (jm(q3) + c) * (b + dn(q2))) * R("h12")
        d1 = dn(q1)
        h = h + ((c + ip(c)) * (ip(a) + ip(d1)) - (im(c) + c) * (a + d1)) * R("h1")
        h = h + 0.25 * ((c + u3) ** 2 - (c + dn(q3)) ** 2) * c3
        H3 = -h
        fp, fm = c3 * m3, c3 * self.col(self.m3, 0, nz - 1)
        D3 = (ip(c) - 2.0 * c + im(c)) * R("s1") + (u3 - c) * fp - (c - dn(q3)) * fm + \
            (no(q3) - c) * R("s3n") - (c - jm(q3)) * R("s3s")
        r = []
        beta = 0.5 * al * dt / Re
        mth = torch.arange(nt // 2 + 1, dtype=F64, device=self.dev) * (2.0 * math.pi / nt)
        for n, (H, D, s) in enumerate(((H1, D1, "s1"), (H2, D2, "s2"), (H3, D3, "s1"))):
            x = (ga * H + ro * self.ru[n][k, j] - al * self.prg[n][k, j] + al / Re * D) * dt
            self.ru[n][k, j] = H
            eig = 1.0 + 2.0 * beta * R(s) * (1.0 - torch.cos(mth))
            r.append(torch.fft.irfft(torch.fft.rfft(x, dim=2) / eig, n=nt, dim=2))
        del H1, H2, H3, D1, D2, D3, h, x

        # ---- outlet and inlet conditions ----
        c3s = (_profile(t + dt) - _profile(t)) * al
        cor = c3s * float(self.da[1:][self.inlet[1:nr + 1]].sum()) * nt / \
            (float((self.qc[1:nr + 1] ** 2 * self.da[1:]).sum()) * nt + float(np.float32(1e-15)))
        qn, qm = q3[nz + 1], q3[nz]
        cs = self.csort.clone()
        cs[1:nr + 1] = torch.where(qn[1:nr + 1] > 0.0, float(np.float32(0.6)) * qn[1:nr + 1], cs[1:nr + 1])
        self.csort = cs
        tconv = -(cs * float(self.m3[nz])) * (qn - qm)
        corr3n = (ga * tconv + ro * self.dq3no) * dt + torch.tensor(self.qc, dtype=F64, device=self.dev)[:, None] * cor
        self.dq3no = tconv

        # ---- implicit r and z sweeps ----
        V = v
        J = np.arange(1, nr + 1)
        lo, hi = beta * V["s1c"][J] * V["s1s"][J], beta * V["s1c"][J] * V["s1n"][J]
        dg = 1.0 + (lo + hi) / rm[J]
        dg[0] = 1.0 + hi[0] / rm[1]
        dg[-1] = 1.0 + lo[-1] / rm[nr] + beta * V["s1c"][nr] * rc[nr + 1] ** 3 / rm[nr + 1]  # slip = 0
        hi1 = -hi / rm[J + 1]
        lo1 = -lo / np.where(J > 1, rm[J - 1], 1.0)
        r[0] = self._inverse(lo1, dg, hi1, 1)(r[0])
        lo, hi = beta * V["s3s"][J] * (J > 1), beta * V["s3n"][J]
        r[2] = self._inverse(-lo, 1.0 + lo + hi, -hi, 1)(r[2])
        kk = np.arange(1, nz + 1)
        ends = ((0.0, 1.0, 0.0), (1.0, 1.0, 0.0))
        zc = np.zeros((3, nz + 1))
        wm, wp = self.m3[kk] * self.c3[kk], self.m3[kk] * self.c3[kk + 1]
        zc[0, :nz], zc[1, :nz], zc[2, :nz] = -beta * wm, 1.0 + beta * (wm + wp), -beta * wp
        zc[:, 0] = 0.0, 1.0 + beta * (self.ws + self.w2), -beta * self.w2
        zc[:, nz] = ends[1]
        zf = np.zeros((3, nz + 1))
        wm, wp = self.c3[kk] * self.m3[kk - 1], self.c3[kk] * self.m3[kk]
        zf[0, :nz], zf[1, :nz], zf[2, :nz] = -beta * wm, 1.0 + beta * (wm + wp), -beta * wp
        zf[:, 0] = zf[:, nz] = ends[0]
        solve_c, solve_f = self._inverse(*zc, 0), self._inverse(*zf, 0)
        dq = [torch.zeros_like(q1) for _ in range(3)]
        K = slice(1, nz + 2)
        zero = torch.zeros(1, nr, nt, dtype=F64, device=self.dev)
        x = torch.cat([zero, r[0][1:], zero])
        dq[0][K, j] = q1[K, j] + solve_c(x)
        x = torch.cat([torch.tensor(self.inlet[1:nr + 1] * c3s, dtype=F64, device=self.dev)[None, :, None].expand(1, nr, nt),
                       r[2][1:], corr3n[None, j]])
        dq[2][K, j] = q3[K, j] + solve_f(x)
        x = torch.cat([zero, r[1][1:], zero])
        x = solve_c(x)
        x[:, 0] = 0.0
        x = torch.cat([x, torch.zeros(nz + 1, 1, nt, dtype=F64, device=self.dev)], dim=1)
        J2 = np.arange(2, nr + 1)
        lo, dg, hi = np.zeros(nr + 1), np.ones(nr + 1), np.zeros(nr + 1)
        lo[1:nr], hi[1:nr] = -beta * V["s2m"][J2], -beta * V["s2p"][J2]
        dg[1:nr] -= lo[1:nr] + hi[1:nr]
        x = self._inverse(lo, dg, hi, 1)(x)
        dq[1][K, j] = q2[K, j] + x[:, :nr]
        del x, r

        # ---- pressure ----
        d = ((ip(dq[0][k, j]) - dq[0][k, j]) * dx1 + (no(dq[1]) - dq[1][k, j]) * dx2) * irm + \
            (up(dq[2]) - dq[2][k, j]) * m3
        ph = torch.zeros_like(q1)
        ph[k, j] = self.poisson(-d / (al * dt))
        del d
        ph[nz + 1] = ph[nz]

        # ---- projection ----
        adt = al * dt
        p = ph[K, j]
        q1[K, j] = dq[0][K, j] - adt * dx1 * irm * (p - im(p))
        q1[K, nr + 1] = 0.0
        rct = torch.tensor(rc, dtype=F64, device=self.dev)[None, :, None]
        q2[K, 2:nr + 1] = dq[1][K, 2:nr + 1] - adt * dx2 * rct[:, 2:nr + 1] * (p[:, 1:] - p[:, :-1])
        q2[K, 1] = 0.0
        q2[K, nr + 1] = 0.0
        q3[1] = dq[2][1]
        K2 = slice(2, nz + 2)
        q3[K2, j] = dq[2][K2, j] - adt * self.col(self.c3, 2, nz + 1) * (ph[K2, j] - ph[k, j])
        q3[K2, nr + 1] = 0.0

        p = ph[k, j]
        pu, pd = up(ph), dn(ph)
        last = torch.zeros(nz, 1, 1, dtype=torch.bool, device=self.dev)
        last[0] = last[-1] = True  # both end planes are their own lower neighbour
        own = lambda x, y: torch.where(last, x, y)  # noqa: E731
        jp_ = lambda x: torch.cat([x[:, 1:], x[:, -1:]], dim=1)  # noqa: E731
        jm_ = lambda x: torch.cat([x[:, :1], x[:, :-1]], dim=1)  # noqa: E731
        irp, irq = jp_(irm), jm_(irm)
        # theta component
        gth = lambda x, w: (x - im(x)) * dx1 * w  # noqa: E731
        G = gth(p, irm)
        lap = (ip(G) - 2.0 * G + im(G)) * R("s1") + (gth(pu, irm) - G) * cp - (G - own(G, gth(pd, irm))) * cm + \
            ((gth(jp_(p), irp) * irn - G * irm) * R("s1n") - (G * irm - gth(jm_(p), irq) * irq) * R("s1s")) * R("s1c")
        self.prg[0][k, j] += G - beta * lap
        # r component, faces j = 2..nr

        def grad_r(x):
            y = torch.zeros(nz, nr + 2, nt, dtype=F64, device=self.dev)  # faces 0..nr+1
            y[:, 2:nr + 1] = (x[:, 1:] - x[:, :-1]) * dx2 * rct[:, 2:nr + 1]
            return y
        F = grad_r(p)
        G, Fu, Fd = F[:, 1:nr + 1], grad_r(pu)[:, 1:nr + 1], grad_r(pd)[:, 1:nr + 1]
        lap = (ip(G) - 2.0 * G + im(G)) * R("s2") + (Fu - G) * cp - (G - own(G, Fd)) * cm + \
            (F[:, 2:] - G) * R("s2p") - (G - F[:, :nr]) * R("s2m")
        self.prg[1][k, 2:nr + 1] += (G - beta * lap)[:, 1:]
        # z component, faces k = 2..nz
        gz = torch.zeros(nz + 2, nr, nt, dtype=F64, device=self.dev)
        gz[2:nz + 2] = (ph[2:nz + 2, j] - ph[1:nz + 1, j]) * self.col(self.c3, 2, nz + 1)
        G = gz[1:nz + 1]
        lap = (ip(G) - 2.0 * G + im(G)) * R("s1") + (gz[2:] - G) * fp - (G - gz[:nz]) * fm + \
            (jp_(G) - G) * R("s3n") - (G - jm_(G)) * R("s3s")
        self.prg[2][2:nz + 1, j] += (G - beta * lap)[1:]
        lap = (ip(p) + im(p) - 2.0 * p) * R("s1") + (jp_(p) - p) * R("s3n") - (p - jm_(p)) * R("s3s") + \
            (pu - p) * cp - (p - own(p, pd)) * cm
        self.pres[k, j] += p - beta * lap

    def step(self, parts=None):
        self.t += self.dt
        for irk in (1, 2, 3):
            if parts is not None:
                parts.stage(irk, self)
            self.substep(irk, self.t)


class _Trilinear:
    """Tracers with Stokes drag, trilinear velocities, one RK3 stage per substep."""

    def __init__(self, u, st, dev):
        self.u = torch.tensor(u, dtype=F64, device=dev)
        self.st, self.f = st, torch.zeros_like(self.u)
        self.alive = torch.ones(u.shape[0], dtype=torch.bool, device=dev)

    def stage(self, irk, s):
        g, u = s.g, self.u
        ga, ro = s.RK[irk]
        r = torch.sqrt(u[:, 0] ** 2 + u[:, 1] ** 2)
        th = torch.atan2(u[:, 1], u[:, 0])
        th = torch.where(th < 0.0, th + 2.0 * math.pi, th)

        def at(q, ot, orr, oz, scale=False):
            pos = [th / g.dth - ot, r / g.dr - orr, u[:, 2] / g.dz - oz]
            fl = [torch.floor(x) for x in pos]
            w = [x - y for x, y in zip(pos, fl)]
            i0, j0, k0 = fl[0].long(), fl[1].long() + 1, fl[2].long() + 1
            w[1] = torch.where(j0 < 0, 0.0, torch.where(j0 > g.nr, 1.0, w[1]))
            w[2] = torch.where(k0 < 0, 0.0, torch.where(k0 > g.nz + 1, 1.0, w[2]))
            j0, k0 = j0.clamp(0, g.nr), k0.clamp(0, g.nz + 1)
            out = torch.zeros_like(r)
            for c in (0, 1):
                for b in (0, 1):
                    for a in (0, 1):
                        x = q[(k0 + c).clamp(max=g.nz + 2), j0 + b, (i0 + a) % g.nt]
                        if scale:
                            face = (j0 + b - 1).to(F64) * g.dr
                            x = torch.where(face > 1e-12, x / torch.where(face > 1e-12, face, 1.0), 0.0)
                        out += (w[0] if a else 1 - w[0]) * (w[1] if b else 1 - w[1]) * (w[2] if c else 1 - w[2]) * x
            return out
        ut, ur, uz = at(s.q[0], 0.0, 0.5, 0.5), at(s.q[1], 0.5, 0.0, 0.5, True), at(s.q[2], 0.5, 0.5, 0.0)
        sn, cs = u[:, 1] / r, u[:, 0] / r
        vel = torch.stack([-sn * ut + cs * ur, cs * ut + sn * ur, uz], dim=1)
        f = torch.cat([u[:, 3:], (vel - u[:, 3:]) / self.st], dim=1)
        on = self.alive[:, None]
        self.u = torch.where(on, u + s.dt * (ga * f + ro * self.f), u)
        self.f = torch.where(on, f, self.f)
        rn = torch.sqrt(self.u[:, 0] ** 2 + self.u[:, 1] ** 2)
        self.alive &= ~((self.u[:, 2] > g.zmax) | (self.u[:, 2] < 0.0) | (rn > g.rmax))


def _exact_step(case, seed):
    g, q, dt, rings = _flow(case, seed)
    n = g.nt * g.nr * g.nz
    if n > 20000000 or (DEV == "cpu" and n > 600000):
        return None
    s = _Stepper(g, case["Re"], dt, q, DEV)
    parts = None
    if case.get("particles") == "trilinear_rk3":
        st = float(np.float32(np.float32(1.0) / np.float32(18.0)) * np.float32(np.float32(998.0) / np.float32(1.2)))
        parts = _Trilinear(_particles(case, seed, rings), st * (5.0e-6 / 0.02) ** 2 * case["Re"], DEV)
    for _ in range(case["steps"]):
        s.step(parts)
    out = dict(zip(_FIELDS, s.q + [s.pres]))
    if case["np"]:
        # the least-squares particles' 117 rows have no short independent form
        out["u"] = parts.u.cpu().numpy() if parts else None
        out["alive"] = parts.alive.cpu().numpy().astype(np.int32) if parts else None
    return out


def _exact_helmholtz(case, seed):
    g = _Grid(3, case["nr"], case["nz"], stretch=2.0)
    f = torch.tensor(_helmholtz_rhs(case, seed), dtype=F64, device=DEV)
    dz, rm = np.diff(g.zf), g.rm[1:g.nr + 1]
    vol = torch.tensor(dz[:, None] * rm[None, :] * g.dr, dtype=F64, device=DEV)
    f[0] -= (f[0] * vol).sum() / vol.sum()  # slot 0 is m = 0
    # z eigenvectors of the flux form, scaled by the cell heights
    zm = 0.5 * (g.zf[1:] + g.zf[:-1])
    iz = np.concatenate([[0.0], 1.0 / np.diff(zm), [0.0]])
    e = -iz[1:-1] / np.sqrt(dz[:-1] * dz[1:])
    lam, W = np.linalg.eigh(np.diag((iz[:-1] + iz[1:]) / dz) + np.diag(e, 1) + np.diag(e, -1))
    lam[0] = 0.0
    V = torch.tensor(W / np.sqrt(dz)[:, None], dtype=F64, device=DEV)
    b = torch.matmul(V.T.contiguous(), f * vol)  # (slots, q, nr)
    rf = np.arange(g.nr + 1, dtype=float)
    rf[0] = rf[g.nr] = 0.0
    m2 = torch.arange(case["slots"], dtype=F64, device=DEV)[None, None, :] ** 2
    t = lambda a: torch.tensor(a, dtype=F64, device=DEV)  # noqa: E731
    bb = m2 * t(g.dr / rm)[None, :, None] + t(rf[:-1] + rf[1:])[None, :, None] + \
        t(lam)[:, None, None] * t(rm * g.dr)[None, :, None]
    bb[0, g.nr - 1, 0] += 1.0  # the singular system: any solution, its mean goes below
    x = _solve_radial([float(a) for a in -rf[:-1]], bb, [float(a) for a in -rf[1:]], b.permute(1, 2, 0).contiguous())
    p = torch.matmul(V, x.permute(2, 0, 1).contiguous())
    p[0] -= (p[0] * vol).sum() / vol.sum()
    p = p.cpu().numpy()
    return p if case["method"] == "direct" else dict(p=p, iters=None)


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "ensemble":
        return [_exact_step(m, seed * 1000 + n) for n, m in enumerate(_members(case))]
    if kind == "poisson":
        g = _Grid(case["nt"], case["nr"], case["nz"])
        phi = _Poisson(g, case["theta"], DEV)(_poisson_rhs(case, seed))
        return phi.cpu().numpy().T
    return _exact_helmholtz(case, seed)
