"""The work this library does for its users, as measurable cases.

A case is one stretch of what a program over the library does again and
again: the TimeSteps between two outputs of a simulation and the output
itself, one whole short run from loaded fields to final fields, a batch of
ensemble requests, the building of a straight-string initial condition.
Sizes and parameters are those of the programs the command line mirrors
(evolution, mpi_evolution, moore, leapfrog, sor + straight_ic), of bench.py
and of the tests, or generic odd sizes in between.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  lattice, pool or parameters in hand before the call
    run(state)           one pass through the public entry points
    work(case)           bytes and operations the path cannot do without
    exact(case, seed)    the same outputs from plain torch in 64 bits
"""
import ctypes
import math

import numpy as np
import torch

import axions_amd as ax
from axions_amd import abi, pool as axpool
from axions_amd.lattice import lib, sor_params, sor_profile

BOUNDARY = {"periodic": abi.AX_BC_PERIODIC, "fixed": abi.AX_BC_FIXED, "neumann": abi.AX_BC_NEUMANN,
            "absorbing": abi.AX_BC_ABSORBING}
DIAG = ("timestep", "finite", "energy", "gauss_mean", "wound_plaquettes", "string_length", "xi")


def _lattice(name, model, shape, precision, **kw):
    """A simulation case.  `steps` TimeSteps per pass; diagnostics every
    `every` of them, with winding counts if `winding`; output per pass: a
    frame of string crossings (`frame`), the winding field (`field`), or the
    whole run from given fields to final fields (`whole`)."""
    c = {"name": name, "kind": "lattice", "model": model, "nx": shape[0], "ny": shape[1], "nz": shape[2],
         "precision": precision, "xy": "periodic", "z": "periodic", "dx": 0.5, "dt": 0.1, "lam": 2.0, "g": 1.0,
         "alpha": 0.0, "damped": 0, "energy_form": 0, "damp_form": 0, "steps": 20, "every": 20, "winding": True,
         "frame": True, "field": False, "whole": False}
    c.update(kw)
    return c


# evolution.cpp's couplings: global strings, PRS friction with a damping window
PRS = {"lam": 1.0, "g": 0.0, "dt": 0.05, "alpha": 3.0, "damped": 200, "damp_form": 1}


def listed():
    return [
        # a whole short run: fields in, 200 steps with energies, final fields
        # out (the 64^3 x 200 configuration the tests pin); latency counts
        _lattice("whole_64", "ah", (64, 64, 64), 64, steps=200, frame=False, whole=True),
        # the evolution program at its own size: energy and Gauss sum every
        # step, a crossings frame every 5 steps
        _lattice("evolution_101", "ah", (101, 101, 101), 64, steps=5, every=1, winding=False, **PRS),
        # a string-network run with the mpi_evolution program's spacings and
        # energy form on an odd cube (its own is 1001^3)
        _lattice("network_301", "ah", (301, 301, 301), 64, dx=0.25, dt=0.05, lam=1.0, alpha=3.0, damped=200,
                 energy_form=1),
        # the benchmark: 512^3 with energy, Gauss sum and windings every 20
        _lattice("plain_512", "ah", (512, 512, 512), 64),
        # the same in single precision
        _lattice("plain_512_fp32", "ah", (512, 512, 512), 32),
        # the evolution program with absorbing faces at a larger size, with
        # the string length by winding number
        _lattice("absorbing_256", "ah", (256, 256, 256), 64, xy="absorbing", **PRS),
        # winding maps of a lattice with Neumann faces, taken every 10 steps
        _lattice("winding_map_160", "ah", (160, 160, 160), 64, xy="neumann", steps=10, every=10, winding=False,
                 frame=False, field=True),
        # the Moore model as the benchmark runs it
        _lattice("moore_256", "moore", (256, 256, 256), 64, dx=0.7, dt=0.2),
        # the moore program's own flat lattice with fixed faces: energy and
        # Gauss sum every step, an output every 10
        _lattice("moore_201x201x51", "moore", (201, 201, 51), 64, xy="fixed", z="fixed", dx=0.7, dt=0.2, steps=10,
                 every=1, winding=False),
        # the leapfrog program's own lattice: the energy printed every step
        _lattice("leapfrog_200", "global", (200, 200, 200), 64, xy="neumann", dx=0.25, dt=0.1, steps=20, every=1,
                 winding=False),
        # a burst of realizations of uneven size through the ensemble pool
        {"name": "ensemble_24", "kind": "ensemble", "requests": 24, "sizes": "64,96,128", "kept": 64, "precision": 32},
        # a straight string: radial profile by relaxation, then the fields
        {"name": "straight_string", "kind": "string", "points": 5001, "h": 0.02, "max_iter": 6000, "g": 0.5,
         "nx": 101, "ny": 101, "nz": 51},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["ah", "moore", "global", "ensemble", "string"], [10, 5, 3, 2, 1])[0]
    if kind == "ensemble":
        sizes = sorted({_size(rng, 40, 144) for _ in range(rng.randint(2, 4))})
        return {"kind": "ensemble", "requests": rng.randint(6, 28), "sizes": ",".join(map(str, sizes)),
                "kept": sizes[0], "precision": rng.choice([32, 32, 64])}
    if kind == "string":
        return {"kind": "string", "points": _size(rng, 1000, 6000), "h": rng.choice([0.01, 0.02, 0.05]),
                "max_iter": _size(rng, 1000, 6000), "g": rng.choice([0.0, 0.5, 1.0]), "nx": rng.randint(48, 128),
                "ny": rng.randint(48, 128), "nz": rng.randint(32, 64)}
    n = _size(rng, 32, {"ah": 400, "moore": 256, "global": 320}[kind])
    shape = [n, n, n] if rng.random() < 0.4 else [max(16, int(n * rng.uniform(0.6, 1.4))) for _ in range(3)]
    big = n > 160
    kw = {"every": rng.choice([1, 5, 10] if not big else [5, 10, 20]), "winding": rng.random() < 0.6}
    kw["steps"] = max(kw["every"], rng.choice([5, 10, 20]))
    out = rng.choices(["frame", "field", "whole"], [6, 2, 0 if n > 128 else 3])[0]
    kw.update(frame=out == "frame", field=out == "field", whole=out == "whole")
    if kind == "ah":
        if rng.random() < 0.5:
            kw.update(lam=rng.choice([1.0, 2.0]), dx=rng.choice([0.25, 0.5]), dt=0.05, alpha=rng.choice([2.0, 3.0]),
                      damped=rng.choice([0, 100, 200]), damp_form=rng.choice([0, 1]), g=rng.choice([0.0, 0.5, 1.0]))
        kw["xy"] = rng.choices(["periodic", "absorbing", "neumann", "fixed"], [6, 2, 1, 1])[0]
        kw["z"] = "fixed" if kw["xy"] == "fixed" else rng.choices(["periodic", "fixed"], [3, 1])[0] \
            if kw["xy"] != "periodic" else "periodic"
        kw["energy_form"] = 1 if kw.get("g", 1.0) != 0 and rng.random() < 0.3 else 0
    elif kind == "moore":
        kw["xy"] = rng.choices(["periodic", "fixed", "neumann"], [3, 1, 1])[0]
        kw.update(z="periodic" if kw["xy"] == "periodic" else "fixed", dx=0.7, dt=0.2)
    else:
        kw.update(xy=rng.choice(["periodic", "neumann"]), dx=rng.choice([0.25, 0.5, 0.7]), dt=0.1)
    c = _lattice("", kind, shape, rng.choice([64, 64, 32]), **kw)
    del c["name"]
    return c


def _params(c):
    if c["model"] == "moore":
        return ax.moore_params(c["nx"], ny=c["ny"], nz=c["nz"], dx=c["dx"], dt=c["dt"], boundary=BOUNDARY[c["xy"]],
                               precision=c["precision"])
    if c["model"] == "global":
        return ax.global_params(c["nx"], ny=c["ny"], nz=c["nz"], dx=c["dx"], dt=c["dt"], boundary=BOUNDARY[c["xy"]],
                                precision=c["precision"])
    return ax.ah_params(c["nx"], ny=c["ny"], nz=c["nz"], dx=c["dx"], dt=c["dt"], lam=c["lam"], g=c["g"],
                        alpha=c["alpha"], damped_nt=c["damped"], theta_damp_form=c["damp_form"],
                        energy_form=c["energy_form"], precision=c["precision"], boundary=BOUNDARY[c["xy"]],
                        boundary_z=BOUNDARY[c["z"]])


def _requests(c, seed):
    """(seed, n, steps) of an ensemble's requests: steps = 2.5 n, the light-
    crossing time of the box at dx = 0.5, dt = 0.1 (bench.py's ensemble)."""
    rng = np.random.RandomState(seed % (1 << 32))
    sizes = [int(v) for v in c["sizes"].split(",")]
    ns = [c["kept"]] + [sizes[i % len(sizes)] for i in range(1, c["requests"])]
    return [(int(rng.randint(1, 1 << 31)), n, int(2.5 * n)) for n in ns]


def _capacity(c):
    return 3 * c["nx"] * c["ny"] * c["nz"] // 2


def _string_lambda(seed):
    return 0.8 + 0.4 * np.random.RandomState(seed % (1 << 32)).random_sample()


class _Simulation:
    def __init__(self, c, seed):
        self.case = c
        self.lat = ax.Lattice(_params(c))
        self.lat.init_random_phase(seed % (1 << 32))
        if c["whole"]:
            self.fields = self.lat.get_state()
        if c["frame"]:
            # a random field has about 1.2 crossings per site, a network fewer
            self.points = torch.zeros((_capacity(c), 3), dtype=torch.float64, device="cuda")
            self.count = torch.zeros(1, dtype=torch.int64, device="cuda")
            torch.cuda.synchronize()


class _Ensemble:
    def __init__(self, c, seed):
        self.case = c
        self.requests = _requests(c, seed)
        self.pool = axpool.Pool(ax.ah_params(8, precision=c["precision"]), hbm_budget=12 << 30, autotune=1,
                                ic_threads=12)
        for n in sorted({n for _, n, _ in self.requests}):
            self.pool.tune(n)


class _String:
    def __init__(self, c, seed):
        self.case = c
        self.sor = sor_params(nx=c["points"], h=c["h"], max_iter=c["max_iter"], g=c["g"], lam=_string_lambda(seed))
        self.lat = ax.Lattice(ax.ah_params(c["nx"], ny=c["ny"], nz=c["nz"], g=c["g"], boundary=abi.AX_BC_FIXED))


def prepare(case, seed):
    return {"lattice": _Simulation, "ensemble": _Ensemble, "string": _String}[case["kind"]](case, seed)


def _frame(s):
    """The crossings of the current field, left on the GPU in the program's
    buffer, and how many of its rows they are."""
    rc = lib.ax_crossings_noalloc(s.lat.handle, s.points.data_ptr(), s.points.shape[0], s.count.data_ptr())
    if rc:
        raise RuntimeError(lib.ax_last_error().decode())
    s.lat.sync()
    return {"count": int(s.count), "points": s.points}


def _simulate(s):
    c, lat, out = s.case, s.lat, {}
    if c["whole"]:
        lat.set_state(s.fields)
    if c["every"] == 1:
        # as the programs' loops: the sums before each step (leapfrog: after it)
        diags = []
        for _ in range(c["steps"]):
            if c["model"] == "global":
                lat.step(1)
            diags.append(lat.diagnostics(winding=c["winding"]))
            if c["model"] != "global":
                lat.step(1)
    else:
        diags = lat.step_diag(c["steps"], c["every"], winding=c["winding"])
    out["diag"] = {k: np.array([d[k] for d in diags]) for k in DIAG}
    if c["frame"]:
        out["frame"] = _frame(s)
    if c["field"]:
        out["winding"] = lat.winding()
    if c["whole"]:
        out["state"] = lat.get_state()
    return out


def _serve(s):
    ids = [s.pool.submit(seed, n, steps, keep_state=i == 0) for i, (seed, n, steps) in enumerate(s.requests)]
    s.pool.wait()
    series = [s.pool.xi(i) for i in ids]
    state = s.pool.get_state(ids[0])
    for i in ids:
        s.pool.release(i)
    return {"timestep": np.concatenate([t for t, _, _ in series]), "wound": np.concatenate([w for _, w, _ in series]),
            "xi": np.concatenate([x for _, _, x in series]), "state": state}


def _straight(s):
    profile, sweeps, residual = sor_profile(s.sor)
    off = s.lat.init_straight_string(profile, s.case["h"])
    return {"profile": profile, "sweeps": sweeps, "residual": residual, "off_grid": off, "state": s.lat.get_state()}


def run(state):
    return {"lattice": _simulate, "ensemble": _serve, "string": _straight}[state.case["kind"]](state)


def work(case):
    if case["kind"] == "string":
        sweeps = case["max_iter"] * case["points"]
        sites = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 32.0 * case["points"] + 2 * 80.0 * sites, "flops": 45.0 * sweeps}
    if case["kind"] == "ensemble":
        updates = float(sum(n ** 3 * t for _, n, t in _requests(case, 0)))
        es = case["precision"] // 8
        return {"bytes": 15.0 * es * updates, "flops": 450.0 * updates}
    sites = float(case["nx"] * case["ny"] * case["nz"])
    es = case["precision"] // 8
    # values read and written per site-update; sines, cosines and products
    values, flops = {"ah": (15, 450.0), "moore": (21, 900.0), "global": (8, 45.0)}[case["model"]]
    b, f = values * es * sites * case["steps"], flops * sites * case["steps"]
    if case["frame"]:
        b += (2 * es + 8) * sites      # phi in, a point for about every third site out
    if case["field"]:
        b += (5 * es + 3) * sites
    if case["whole"]:
        levels = {"ah": 10, "moore": 14, "global": 4}[case["model"]]
        b += 2 * 8 * levels * sites    # host fields in and out
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# The same outputs from plain torch in double precision.
# ---------------------------------------------------------------------------
def _up(f, a):
    return torch.roll(f, -1, a)        # f at s + a


def _dn(f, a):
    return torch.roll(f, 1, a)         # f at s - a


def _phases(seed, n):
    """std::uniform_real_distribution(0, 2 pi) over std::mt19937(seed)."""
    u = np.random.RandomState(seed % (1 << 32)).randint(0, 1 << 32, size=2 * n, dtype=np.uint32).reshape(n, 2)
    return (u[:, 0] + u[:, 1] * 4294967296.0) * (2 * math.pi / 18446744073709551616.0)


def _initial(seed, shape, fields, dev):
    n = int(np.prod(shape))
    ph = torch.from_numpy(_phases(seed, n * fields)).to(dev).reshape(*shape, fields)
    out = []
    for f in range(fields):
        out += [torch.cos(ph[..., f]).contiguous(), torch.sin(ph[..., f]).contiguous()]
    return out


class _Exact:
    """Gauged lattices (one or two scalars on one U(1) link field)."""

    def __init__(self, c, shape, phi):
        self.c, self.shape = c, shape
        p = self.p = _params(c)
        self.q = [1.0] if c["model"] == "ah" else [float(p.q1), float(p.q2)]
        zero = torch.zeros_like(phi[0])
        self.cur = phi + [zero.clone() for _ in range(3)]
        self.prv = [x.clone() for x in self.cur]
        self.d = [p.dx, p.dy, p.dz]
        self.n = 0
        self.inner = torch.ones(shape, dtype=torch.bool, device=zero.device)
        for a in range(3):
            if c["xy" if a < 2 else "z"] != "periodic":
                self.inner.narrow(a, 0, 1).fill_(False)
                self.inner.narrow(a, shape[a] - 1, 1).fill_(False)

    def potentials(self):
        p = self.p
        m = [self.cur[2 * f] ** 2 + self.cur[2 * f + 1] ** 2 for f in range(len(self.q))]
        if len(m) == 1:
            w = m[0] - p.eta ** 2
            return [0.5 * p.lambda_ * w], 0.25 * p.lambda_ * w * w
        w1, w2 = m[0] - p.eta1 ** 2, m[1] - p.eta2 ** 2
        return ([0.5 * (p.lambda1 * w1 + p.lambda12 * w2), 0.5 * (p.lambda2 * w2 + p.lambda12 * w1)],
                0.25 * p.lambda1 * w1 * w1 + 0.25 * p.lambda2 * w2 * w2 + 0.5 * p.lambda12 * w1 * w2)

    def angle(self, a, b):
        t = self.cur[-3:]
        return t[a] + _up(t[b], a) - _up(t[a], b) - t[b]

    def step(self):
        p, t, g = self.p, self.cur[-3:], self.p.g
        damp = p.dampFac if self.n < p.damped_nt else 0.0
        fric = damp + p.alpha * p.scaling / (1 + self.n * p.dt)
        moore = self.c["model"] == "moore"
        pots, _ = self.potentials()
        new, force = [], [0.0, 0.0, 0.0]
        for f, q in enumerate(self.q):
            r, i = self.cur[2 * f], self.cur[2 * f + 1]
            ar, ai = -pots[f] * r, -pots[f] * i
            for a in range(3):
                co, si = torch.cos(q * t[a]), torch.sin(q * t[a])
                rn, in_ = _up(r, a), _up(i, a)
                back_r, back_i = _dn(co * r - si * i, a), _dn(co * i + si * r, a)
                ar += (co * rn + si * in_ - 2 * r + back_r) / self.d[a] ** 2
                ai += (co * in_ - si * rn - 2 * i + back_i) / self.d[a] ** 2
                force[a] = force[a] - 2 * g * g * q * (co * (i * rn - r * in_) + si * (r * rn + i * in_))
            for k, acc in ((2 * f, ar), (2 * f + 1, ai)):
                if not moore:
                    acc -= fric * (self.cur[k] - self.prv[k]) / p.dt
                new.append(2 * self.cur[k] - self.prv[k] + p.dt ** 2 * acc)
        for a in range(3):
            for b in range(3):
                if a != b:
                    s = torch.sin(self.angle(a, b))
                    force[a] = force[a] - (s - _dn(s, b)) / self.d[b] ** 2
            k = len(self.cur) - 3 + a
            if not moore:
                force[a] = force[a] - damp * (self.cur[k] - self.prv[k]) / p.dt
            new.append(2 * self.cur[k] - self.prv[k] + p.dt ** 2 * force[a])
        if not bool(self.inner.all()):
            new = [torch.where(self.inner, x, o) for x, o in zip(new, self.prv)]
        self.prv, self.cur = self.cur, new
        self.n += 1

    def diag(self, winding):
        p, t, g, dt = self.p, self.cur[-3:], self.p.g, self.p.dt
        old = self.prv[-3:]
        charge = 0.0
        rho = self.potentials()[1]
        for f, q in enumerate(self.q):
            r, i = self.cur[2 * f], self.cur[2 * f + 1]
            vr, vi = (r - self.prv[2 * f]) / dt, (i - self.prv[2 * f + 1]) / dt
            rho = rho + vr * vr + vi * vi
            charge = charge + q * (i * vr - r * vi)
            for a in range(3):
                co, si = torch.cos(q * t[a]), torch.sin(q * t[a])
                rho = rho + ((r - _dn(co * r - si * i, a)) / self.d[a]) ** 2
                rho = rho + ((i - _dn(co * i + si * r, a)) / self.d[a]) ** 2
        gauss = torch.zeros_like(rho)
        if g != 0:
            for a in range(3):
                e = (t[a] - old[a]) / dt if p.energy_form == 1 else (t[a] - old[a]) / (g * dt * self.d[a])
                rho = rho + 0.5 * e * e
                for b in range(a + 1, 3):
                    rho = rho + (1 - torch.cos(self.angle(a, b))) / (g * self.d[a] * self.d[b]) ** 2
                rate = (t[a] - old[a]) / dt
                gauss = gauss + (rate - _dn(rate, a)) / (g * self.d[a] ** 2)
            gauss = (gauss - 2 * g * charge).abs()
        sums = [float((x * self.inner).sum()) for x in (rho, gauss)]
        open_xy, open_z = self.c["xy"] != "periodic", self.c["z"] != "periodic"
        nx, ny, nz = self.shape
        sites = (nx - 2 * open_xy) * (ny - 2 * open_xy) * (nz - 2 * open_z)
        no_gauss = self.c["model"] == "ah" and p.energy_form == 1
        out = {"timestep": self.n, "finite": 1, "energy": sums[0] * self.d[0] * self.d[1] * self.d[2],
               "gauss_mean": 0.0 if no_gauss else sums[1] / sites}
        out.update(_wound(self.cur[0], self.cur[1], t, self.q[0], self.d, (open_xy, open_xy, open_z), winding))
        return out

    def winding(self):
        open_xy, open_z = self.c["xy"] != "periodic", self.c["z"] != "periodic"
        return torch.stack(_winding(self.cur[0], self.cur[1], self.cur[-3:], self.q[0], (open_xy, open_xy, open_z)))

    def phi(self):
        return self.cur[0], self.cur[1]

    def open(self):
        return self.c["xy"] != "periodic", self.c["z"] != "periodic"

    def state(self):
        levels = {(self.n + 1) % 2: self.cur, self.n % 2: self.prv}
        return torch.stack([levels[k][f] for f in range(len(self.cur)) for k in (0, 1)]).reshape(-1)


def _winding(r, i, t, q, opened):
    z = torch.complex(r, i)
    edge = [torch.angle(z.conj() * torch.exp(-1j * q * t[a]) * _up(z, a)) for a in range(3)]
    out = []
    for a, b in ((0, 1), (0, 2), (1, 2)):
        e = [edge[k] + q * t[k] for k in (a, b)]
        w = torch.round((e[0] + _up(e[1], a) - _up(e[0], b) - e[1]) / (2 * math.pi)).to(torch.int8)
        for k in (a, b):
            if opened[k]:
                w.narrow(k, w.shape[k] - 1, 1).zero_()
        out.append(w)
    return out


def _wound(r, i, t, q, d, opened, winding):
    if not winding:
        return {"wound_plaquettes": 0, "string_length": 0.0, "xi": 0.0}
    n = [int(w.abs().sum(dtype=torch.int64)) for w in _winding(r, i, t, q, opened)]
    length = (2.0 / 3.0) * (n[0] * d[2] + n[1] * d[1] + n[2] * d[0])
    return {"wound_plaquettes": sum(n), "string_length": length, "xi": length / (r.numel() * d[0] * d[1] * d[2])}


class _ExactGlobal:
    """leapfrog.cpp: momentum form, no gauge field."""

    def __init__(self, c, shape, phi):
        self.c, self.shape, self.p = c, shape, _params(c)
        self.f, self.m = phi, [torch.zeros_like(x) for x in phi]
        self.old, self.n = None, 0
        self.inner = torch.ones(shape, dtype=torch.bool, device=phi[0].device)
        if c["xy"] != "periodic":
            for a in (0, 1):
                self.inner.narrow(a, 0, 1).fill_(False)
                self.inner.narrow(a, shape[a] - 1, 1).fill_(False)

    def acceleration(self):
        mag = self.f[0] ** 2 + self.f[1] ** 2
        d = (self.p.dx, self.p.dy, self.p.dz)
        return [sum((_up(x, a) - 2 * x + _dn(x, a)) / d[a] ** 2 for a in range(3)) - (mag - 1) * x for x in self.f]

    def step(self):
        if self.c["xy"] != "periodic":
            nx, ny = self.shape[:2]
            for x in self.f:
                x[:, 0], x[:, ny - 1] = x[:, 1].clone(), x[:, ny - 2].clone()
                x[0], x[nx - 1] = x[1].clone(), x[nx - 2].clone()
        self.acc = self.acceleration()
        self.old = self.f
        self.m = [torch.where(self.inner, m + a * self.p.dt, m) for m, a in zip(self.m, self.acc)]
        self.f = [torch.where(self.inner, x + m * self.p.dt, x) for x, m in zip(self.f, self.m)]
        self.n += 1

    def diag(self, winding):
        out = {"timestep": self.n, "finite": 1, "energy": math.nan, "gauss_mean": 0.0}
        d = (self.p.dx, self.p.dy, self.p.dz)
        if self.n:
            # the sum as the program's one-thread loop prints it: neighbours
            # earlier in site order already hold their new values
            mag = self.old[0] ** 2 + self.old[1] ** 2
            rho = 0.5 * (mag - 1) ** 2
            for k in (0, 1):
                rho = rho + (self.m[k] - 0.5 * self.acc[k] * self.p.dt) ** 2
                for a in range(3):
                    plus, minus = _up(self.old[k], a), _dn(self.f[k], a)
                    plus.narrow(a, self.shape[a] - 1, 1).copy_(self.f[k].narrow(a, 0, 1))
                    minus.narrow(a, 0, 1).copy_(self.old[k].narrow(a, self.shape[a] - 1, 1))
                    rho = rho + ((plus - minus) / (2 * d[a])) ** 2
            out["energy"] = float((rho * self.inner).sum()) * d[0] * d[1] * d[2]
        zero = torch.zeros_like(self.f[0])
        out.update(_wound(self.f[0], self.f[1], [zero] * 3, 0.0, d, (False,) * 3, winding))
        return out

    def winding(self):
        return torch.stack(_winding(self.f[0], self.f[1], [torch.zeros_like(self.f[0])] * 3, 0.0, (False,) * 3))

    def phi(self):
        return self.f

    def open(self):
        return False, False

    def state(self):
        return torch.stack(list(self.f) + list(self.m)).reshape(-1)


def _roots(v00, v10, v01, v11, u, du, w, dw):
    """The zeros of the bilinear interpolation of phi over a face."""
    c1 = [v11[c] - v10[c] - v01[c] + v00[c] for c in (0, 1)]
    c2 = [(w + dw) * (v10[c] - v00[c]) + w * (v01[c] - v11[c]) for c in (0, 1)]
    c3 = [(u + du) * (v01[c] - v00[c]) + u * (v10[c] - v11[c]) for c in (0, 1)]
    c4 = [(u + du) * ((w + dw) * v00[c] - w * v01[c]) - u * ((w + dw) * v10[c] - w * v11[c]) for c in (0, 1)]
    a = c1[1] * c3[0] - c1[0] * c3[1]
    b = c1[1] * c4[0] + c2[1] * c3[0] - c1[0] * c4[1] - c2[0] * c3[1]
    c = c2[1] * c4[0] - c2[0] * c4[1]
    disc = b * b - 4 * a * c
    line = a == 0
    found = []
    for sign in (1.0, -1.0):
        s2 = (-b + sign * torch.sqrt(disc)) / (2 * a)
        ok = ~line & (disc >= 0)
        if sign > 0:
            s2, ok = torch.where(line, -c / b, s2), torch.where(line, b != 0, ok)
        s1 = -(c3[0] * s2 + c4[0]) / (c1[0] * s2 + c2[0])
        found.append((ok & (s2 >= w) & (s2 <= w + dw) & (s1 >= u) & (s1 <= u + du), s1, s2))
    return found


def _crossings(model):
    f, (open_xy, open_z), (nx, ny, nz) = model.phi(), model.open(), model.shape
    d = (model.p.dx, model.p.dy, model.p.dz)
    at = [((torch.arange(n, device=f[0].device, dtype=torch.float64) - int(0.5 * (n - 1))) * h)
          for n, h in zip((nx, ny, nz), d)]
    got = []
    for x0 in range(0, nx, 16):
        ids = torch.arange(x0, min(nx, x0 + 16), device=f[0].device)
        here = [g[ids] for g in f]
        next_ = [g[(ids + 1) % nx] for g in f]
        x, y, z = at[0][ids][:, None, None], at[1][None, :, None], at[2][None, None, :]
        vx, vy, vz = next_, [_up(g, 1) for g in here], [_up(g, 2) for g in here]
        vxy, vxz, vyz = [_up(g, 1) for g in next_], [_up(g, 2) for g in next_], [_up(_up(g, 1), 2) for g in here]
        keep = torch.ones_like(here[0], dtype=torch.bool)
        if open_xy:
            keep &= ((ids > 0) & (ids < nx - 1))[:, None, None]
            keep[:, 0] = keep[:, -1] = False
        if open_z:
            keep[..., 0] = keep[..., -1] = False
        ok, pts = [], []
        for face, (a, b, ab, u, du, w, dw) in enumerate(((vx, vy, vxy, x, d[0], y, d[1]),
                                                         (vx, vz, vxz, x, d[0], z, d[2]),
                                                         (vy, vz, vyz, y, d[1], z, d[2]))):
            for hit, s1, s2 in _roots(here, a, b, ab, u, du, w, dw):
                third = (z, y, x)[face].expand_as(s1)
                ok.append(hit & keep)
                pts.append(torch.stack(((s1, s2, third), (s1, third, s2), (third, s1, s2))[face], -1))
        ok, pts = torch.stack(ok, -1), torch.stack(pts, -2)
        got.append(pts[ok])
    return torch.cat(got)


def _exact_lattice(c, seed):
    if "absorbing" in (c["xy"], c["z"]) or c["xy"] == "neumann" and c["model"] != "global":
        return None                    # face equations of their own
    shape = (c["nx"], c["ny"], c["nz"])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    phi = _initial(seed, shape, 2 if c["model"] == "moore" else 1, dev)
    m = (_ExactGlobal if c["model"] == "global" else _Exact)(c, shape, phi)
    del phi
    diags = []
    for s in range(c["steps"]):
        if s % c["every"] == 0 and not (c["model"] == "global" and c["every"] == 1):
            diags.append(m.diag(c["winding"]))
        m.step()
        if c["model"] == "global" and c["every"] == 1:
            diags.append(m.diag(c["winding"]))
    out = {"diag": {k: np.array([d[k] for d in diags]) for k in DIAG}}
    if c["frame"]:
        # among very many crossings some lie on the edge of two faces within
        # rounding, and one more or less shifts all that follow in the list
        pts = _crossings(m) if c["precision"] == 64 and m.inner.numel() <= 1 << 23 else None
        out["frame"] = {"count": None, "points": None}
        if pts is not None:
            out["frame"]["count"] = pts.shape[0]
            out["frame"]["points"] = torch.nn.functional.pad(pts, (0, 0, 0, _capacity(c) - pts.shape[0]))
    if c["field"]:
        out["winding"] = m.winding().reshape(-1)
    if c["whole"]:
        out["state"] = m.state()
    return out


def _exact_ensemble(c, seed):
    """The kept realization's final fields; the series count windings."""
    s, n, steps = _requests(c, seed)[0]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    case = _lattice("", "ah", (n, n, n), c["precision"])
    m = _Exact(case, (n, n, n), _initial(s, (n, n, n), 1, dev))
    for _ in range(steps):
        m.step()
    return {"timestep": None, "wound": None, "xi": None, "state": m.state()}


def exact(case, seed):
    if case["kind"] == "lattice":
        return _exact_lattice(case, seed)
    if case["kind"] == "ensemble":
        return _exact_ensemble(case, seed)
    return None                        # thousands of sequential sweeps
