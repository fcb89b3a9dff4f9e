"""Performance cases of the hydro step: what a simulation program has the
library do between two of its outputs.

A pass takes a number of main-loop steps (the device-resident loop, the
per-step calls a host code makes, or a batch of independent boxes) and brings
the state back into the host's padded arrays, as a program does for each
output.  Small boxes start from an upload in every pass (a whole short
simulation); large ones go on from where the last pass left them (one output
interval of a long run).

A case's values: ``kind`` the set-up (tube, vortex, shear, star, ensemble),
``n1, n2, n3`` the cells, ``steps`` the steps of a pass, ``loop`` how they are
taken (device, host or batch), ``load`` whether a pass starts from an upload,
``mag`` MHD or hydro, ``limiter``, ``rk`` the Runge-Kutta order,
``precision``, ``species`` the number of advected species, ``fused`` the
argument of Hydro.set_fused, and ``boxes`` the members of an ensemble.
"""
import math

import numpy as np
import torch

from hormone_amd import driver as D
from hormone_amd import problems as P
from hormone_amd.batch import Batch
from hormone_amd.grid import cartesian_grid
from hormone_amd.native import Hydro

NEVER = 1 << 40


def _case(name, kind, n1, n2, n3, steps, **kw):
    c = {"name": name, "kind": kind, "n1": n1, "n2": n2, "n3": n3, "steps": steps,
         "loop": "device", "load": True, "mag": True, "limiter": "modified_mc", "rk": 3,
         "precision": "fp64", "species": 0, "fused": 0, "boxes": ""}
    c.update(kw)
    return c


def listed():
    return [
        # the reference's Sod test, the smallest box: launches and latency
        _case("sod_x_500", "tube", 500, 1, 1, 300, mag=False),
        # 1D MHD shock tube along the slowest axis, an odd size
        _case("briowu_z_1001", "tube", 1, 1, 1001, 200),
        # the Orszag-Tang vortex at the size of the reference's test
        _case("vortex_xy_128", "vortex", 128, 128, 1, 400),
        # and at benchmark size
        _case("vortex_xy_512", "vortex", 512, 512, 1, 500),
        # 2D hydro shear layer with two advected species (the reference's test)
        _case("shear_species_128", "shear", 128, 128, 1, 300, mag=False, species=2),
        # ragged 3D MHD box, minmod, no extent a multiple of anything
        _case("shear_ragged_130", "shear", 97, 131, 75, 30, load=False, limiter="minmod"),
        # 3D hydro, second-order Runge-Kutta
        _case("shear_hydro_160", "shear", 160, 160, 160, 30, load=False, mag=False, rk=2),
        # 3D MHD turbulence runs: FP64 and the mixed-precision solver
        _case("shear_256", "shear", 256, 256, 256, 40, load=False, fused=2),
        _case("shear_mixed_192", "shear", 192, 192, 192, 40, load=False, fused=2,
              precision="fp32mix"),
        # self-gravitating star, the benchmark workload
        _case("star_256", "star", 256, 256, 256, 60, load=False, fused=2),
        # the same driven call by call from a host code's own main loop
        _case("star_host_128", "star", 128, 128, 128, 20, load=False, loop="host", fused=2),
        # a serving batch of 2D and 3D requests
        _case("ensemble_8", "ensemble", 0, 0, 0, 100, loop="batch",
              boxes="64x64x1,101x101x1,150x150x1,192x192x1,36x36x36,48x48x48,63x63x63,80x80x80"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("tube", "vortex", "shear", "shear", "star", "ensemble"))
    if kind == "tube":
        n = [1, 1, 1]
        n[rng.randrange(3)] = _log_int(rng, 100, 4096)
        return _unnamed("tube", *n, rng.randint(100, 300), mag=rng.random() < 0.5,
                        limiter=rng.choice(("modified_mc", "minmod")), rk=rng.choice((2, 3)))
    if kind == "vortex":
        m = _log_int(rng, 48, 640)
        n = rng.choice(((m, m, 1), (m, 1, m), (1, m, m)))
        return _unnamed("vortex", *n, rng.randint(100, 300))
    if kind == "ensemble":
        b = [(_log_int(rng, 64, 192),) * 2 + (1,) for _ in range(rng.randint(2, 5))]
        b += [(_log_int(rng, 34, 90),) * 3 for _ in range(rng.randint(1, 4))]
        return _unnamed("ensemble", 0, 0, 0, rng.randint(40, 100), loop="batch",
                        boxes=",".join("%dx%dx%d" % x for x in b))
    m = _log_int(rng, 40, 220)
    if kind == "star":
        m = min(m, 190)
        return _unnamed("star", m, m, m, rng.randint(10, 30), load=m < 100, mag=rng.random() < 0.7,
                        fused=rng.choice((0, 2)), loop=rng.choice(("device", "device", "host")))
    n = [max(20, int(m * rng.uniform(0.7, 1.2))) for _ in range(3)]
    if rng.random() < 0.25:
        return _unnamed("shear", 2 * n[0], 2 * n[1], 1, rng.randint(60, 200), mag=False,
                        species=rng.randint(1, 3))
    return _unnamed("shear", *n, rng.randint(10, 40), load=m < 100, mag=rng.random() < 0.7,
                    limiter=rng.choice(("modified_mc", "minmod", "flat")), rk=rng.choice((2, 3, 3)),
                    precision=rng.choice(("fp64", "fp64", "fp32mix")), fused=rng.choice((0, 2)))


def _unnamed(*a, **kw):
    c = _case("", *a, **kw)
    del c["name"]
    return c


# ---- inputs -----------------------------------------------------------------

def _params(case, n):
    """The run's settings (hormone_amd.problems.Params)."""
    free = case["kind"] in ("tube", "star", "ensemble")
    p = P.Params(n=n, mag_on=case["mag"], flux_limiter=case["limiter"], rktype=case["rk"],
                 precision=case["precision"], bc=((3,) * 12 if free else (0,) * 12),
                 outstyle=2, endstyle=2, tnlim=NEVER, tn_out=NEVER, t_end=1e30, is_test=False)
    if case["kind"] == "tube":
        p.gamma = 2.0 if case["mag"] else 1.4
    if case["kind"] == "star":
        p.gamma, p.gravswitch, p.G = 2.0, 3, 1.0
        p.lo, p.hi = (-1.0,) * 3, (1.0,) * 3
    if case["species"]:
        p.compswitch, p.spn = 2, case["species"]
    return p


def _fields(case, n, prm, seed):
    """Initial primitives as (nz, ny, nx) float64 tensors, every value from
    the seed: d, p, v, b and, where the set-up has them, spc and grvphi (with
    two ghost layers)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    r = np.random.default_rng(seed)
    shape = (n[2], n[1], n[0])
    one = torch.ones(shape, dtype=torch.float64, device=dev)

    def centre(a, pad=0):
        h = (prm.hi[a] - prm.lo[a]) / n[a]
        x = prm.lo[a] + h * (torch.arange(-pad, n[a] + pad, dtype=torch.float64, device=dev) + 0.5)
        return x.reshape([-1 if 2 - a == q else 1 for q in range(3)])

    def noise():
        return 2.0 * torch.rand(shape, generator=gen, dtype=torch.float64, device=dev) - 1.0

    v, b, out = [0.0 * one for _ in range(3)], [0.0 * one for _ in range(3)], {}
    kind = case["kind"]
    if kind == "tube":  # Sod or Brio-Wu like states, each side jittered
        a = next(q for q in range(3) if n[q] > 1)
        left = (centre(a) < 0.5).expand(shape)
        j = 1.0 + 0.1 * r.uniform(-1, 1, 8)
        d = torch.where(left, 1.0 * j[0], 0.125 * j[1]) * one
        p = torch.where(left, 1.0 * j[2], 0.1 * j[3]) * one
        if case["mag"]:
            b[a] = 0.75 * j[4] * one
            b[(a + 1) % 3] = torch.where(left, 1.0 * j[5], -1.0 * j[6]) * one
    elif kind == "vortex":  # Orszag-Tang in the solved plane
        a, c = [q for q in range(3) if n[q] > 1]
        j = 1.0 + 0.05 * r.uniform(-1, 1, 6)
        tau, s4 = 2.0 * math.pi, math.sqrt(4.0 * math.pi)
        d = prm.gamma ** 2 / (4.0 * math.pi) * j[0] * one
        p = prm.gamma / (4.0 * math.pi) * j[1] * one
        v[a] = -j[2] * torch.sin(tau * centre(c)) * one
        v[c] = j[3] * torch.sin(tau * centre(a)) * one
        b[a] = -j[4] * torch.sin(tau * centre(c)) / s4 * one
        b[c] = j[5] * torch.sin(2.0 * tau * centre(a)) / s4 * one
    elif kind == "shear":  # Kelvin-Helmholtz layer with a noisy cross flow
        inside = ((centre(1) - 0.5).abs() < 0.25).expand(shape)
        d = torch.where(inside, 1.0, 2.0) * one
        p = 2.5 * one
        v[0] = torch.where(inside, 0.5, -0.5) * one
        v[1] = 0.01 * noise() * torch.sin(4.0 * math.pi * centre(0))
        if case["mag"]:
            b[0] = 0.1 * one
        if case["species"]:
            s = torch.where(inside, 0.1, 0.9) * one
            share = [s] + [(1.0 - s) / max(1, case["species"] - 1)] * (case["species"] - 1)
            out["spc"] = share if case["species"] > 1 else [one]
    elif kind == "star":  # n=1 polytrope (M = G = 1, R = 0.3) in a thin background
        R, bg = 0.3, 1e-6
        rho_c, K = math.pi / (4.0 * R ** 3), 2.0 * R * R / math.pi

        def rho(rad):
            return torch.where(rad < R, rho_c * torch.sinc(rad / R), 0.0)

        def radius(pad):
            return torch.sqrt(sum(centre(q, pad) ** 2 for q in range(3)))
        star = rho(radius(0))
        p = K * star * star + bg / torch.clamp(radius(0), min=R)
        d = torch.clamp(star, min=bg) * (1.0 + 1e-3 * noise())
        rad = radius(2)
        out["grvphi"] = torch.where(rad < R, -1.0 / R - 2.0 * K * rho(rad), -1.0 / rad)
    else:  # ensemble member: Riemann problem or blast, states drawn per request
        rho, pr = r.lognormal(0.0, 0.5, 2), r.lognormal(0.0, 0.5, 2)
        left = (centre(0) < 0.5).expand(shape)
        d = torch.where(left, rho[0], rho[1]) * one
        p = torch.where(left, pr[0], pr[1]) * one
        if r.uniform() < 0.5:
            r2 = sum((centre(q) - 0.5) ** 2 for q in range(3) if n[q] > 1)
            d = rho[0] * one
            p = torch.where((r2 < 0.01).expand(shape), 5.0 * pr.max(), pr[1]) * one
        v = [x * one for x in r.uniform(-0.5, 0.5, 3)]
        b = [x * one for x in r.uniform(-0.5, 0.5, 3)]
    out.update(d=d, p=p, v=v, b=b)
    return out


def _uploads(case, prm, g, f):
    """(field, padded host array) of every upload that starts a run."""
    d, (v1, v2, v3), (b1, b2, b3) = f["d"], f["v"], f["b"]
    e = (f["p"] / (prm.gamma - 1.0) + (d * 0.5) * ((v1 * v1 + v2 * v2) + v3 * v3)) \
        + 0.5 * ((b1 * b1 + b2 * b2) + b3 * b3)
    zero = torch.zeros_like(d)
    todo = [(D.F_D, d), (D.F_V1, v1), (D.F_V2, v2), (D.F_V3, v3), (D.F_E, e)]
    u = [d, d * v1, d * v2, d * v3, e]
    if prm.mag_on:
        todo += [(D.F_B1, b1), (D.F_B2, b2), (D.F_B3, b3), (D.F_PHI, zero)]
        u += [b1, b2, b3] + ([zero] if g.dim > 1 else [])
    todo += [(D.F_U + q, a) for q, a in enumerate(u)]
    todo += [(D.F_SPC + q, a) for q, a in enumerate(f.get("spc", ()))]
    if prm.gravswitch == 3:
        todo.append((D.F_GRVPSI, zero))

    def padded(a):
        h = np.zeros(g.padded_shape)
        h[2:-2, 2:-2, 2:-2] = a.cpu().numpy()
        return h
    for field, a in todo:
        yield field, padded(a)
    if prm.gravswitch == 3:
        yield D.F_GRVPHI, f["grvphi"].cpu().numpy()


class _Sim:
    """One simulation as a host program holds it: the context, its host
    arrays and its clock."""

    def __init__(self, case, n, seed, load):
        self.prm = _params(case, n)
        self.g = cartesian_grid(n, self.prm.lo, self.prm.hi, gravity=self.prm.gravswitch == 3)
        self.eng = Hydro(**D.desc_fields(self.prm, self.g))
        if case["fused"]:
            self.eng.set_fused(case["fused"])
        ups = _uploads(case, self.prm, self.g, _fields(case, n, self.prm, seed))
        self.ups = list(ups) if load else None
        if not load:
            for field, a in ups:
                self.eng.upload(field, a)
        fields = list(D.SNAP_FIELDS_MAG if self.prm.mag_on else D.SNAP_FIELDS)
        fields += [D.F_SPC + q for q in range(case["species"])]
        if self.prm.gravswitch == 3:
            fields += [D.F_GRVPHI, D.F_GRVPSI]
        self.block = np.zeros((len(fields),) + self.g.padded_shape)
        self.host = dict(zip(fields, self.block))
        self.damp = math.exp(-self.prm.alpha9wave * self.prm.courant) \
            if self.prm.mag_on and self.g.dim > 1 else 0.0
        self.restart()

    def restart(self):
        self.time, self.tn, self.grvtime, self.cgrav_old = 0.0, 0, 0.0, 0.0

    def upload(self):
        for field, a in self.ups:
            self.eng.upload(field, a)
        self.restart()

    def download(self):
        for field, a in self.host.items():
            self.eng.download(field, a)

    def device_loop(self, steps):
        if self.prm.gravswitch == 3:
            self.time, self.tn, _, _, self.grvtime, self.cgrav_old, _ = self.eng.run_loop_gravity(
                self.time, self.tn, 1e30, 1e30, 1e30, 2, 2, NEVER, NEVER, steps, self.damp,
                self.grvtime, self.cgrav_old)
        else:
            self.time, self.tn, _, _ = self.eng.run_loop(
                self.time, self.tn, 1e30, 1e30, 1e30, 2, 2, NEVER, NEVER, steps, self.damp)

    def host_loop(self, steps):
        """hormone.f90's main loop, call by call."""
        eng = self.eng
        for _ in range(steps):
            if self.prm.gravswitch == 3:
                dt, ch, cgrav, dtgrav = eng.timestep(self.time, 1e30, 1e30, 2, 2, grav=True)
                if self.tn == 0:
                    self.grvtime = 0.0
                else:
                    self.grvtime, self.cgrav_old, dtgrav, _ = eng.gravity(
                        self.time, dt, self.grvtime, cgrav, self.cgrav_old, dtgrav)
            else:
                dt, ch = eng.timestep(self.time, 1e30, 1e30, 2, 2)
            eng.hydro_step(dt, ch)
            if self.damp > 0.0:
                eng.phidamp(self.damp)
            self.time += dt
            self.tn += 1


def _sizes(case):
    if case["loop"] == "batch":
        return [tuple(int(x) for x in b.split("x")) for b in case["boxes"].split(",")]
    return [(case["n1"], case["n2"], case["n3"])]


def prepare(case, seed):
    sims = [_Sim(case, n, seed + 1000 * q, case["load"]) for q, n in enumerate(_sizes(case))]
    return {"case": case, "sims": sims, "batch": Batch() if case["loop"] == "batch" else None}


def run(state):
    case, sims, batch = state["case"], state["sims"], state["batch"]
    if case["load"]:
        for s in sims:
            s.upload()
    if batch is not None:
        for s in sims:
            batch.add(s.eng, t_end=1e30, t_out=1e30, dt_out=1e30, outstyle=2, endstyle=2,
                      tnlim=NEVER, tn_out=NEVER)
        batch.step(case["steps"])
        for s in sims:
            s.time, s.tn, _ = batch.state(s.eng)
            batch.remove(s.eng)
    elif case["loop"] == "host":
        sims[0].host_loop(case["steps"])
    else:
        sims[0].device_loop(case["steps"])
    for s in sims:
        s.download()
    # every field an output of its own; an ensemble's, one block per member
    return [{"time": s.time, "tn": s.tn,
             "fields": s.block if batch is not None else list(s.host.values())} for s in sims]


def work(case):
    """Per step and stage every conserved field is read and written once (from
    stage 2 on the step's start is read as well); about 700 (MHD) or 300
    (hydro) operations per cell, direction and stage; six gravity sub-steps a
    step, each reading potential, its rate and density and writing two.  Each
    upload and download once."""
    nbytes = flops = 0.0
    for n in _sizes(case):
        cells = n[0] * n[1] * n[2]
        dim = sum(x > 1 for x in n)
        nv = (9 if dim > 1 else 8) if case["mag"] else 5
        nv += case["species"]
        io = (2 * nv if case["load"] else 0) + nv
        nbytes += 8.0 * cells * (case["steps"] * nv * (3 * case["rk"] - 1) + io)
        flops += cells * case["steps"] * case["rk"] * dim * (700.0 if case["mag"] else 300.0)
        if case["kind"] == "star":
            nbytes += 8.0 * cells * case["steps"] * 6 * 5
            flops += cells * case["steps"] * 6 * 60.0
    return {"bytes": nbytes, "flops": flops}


# ---- the same steps in plain torch, 64 bits ------------------------------------
# Written from the scheme (MUSCL on conserved variables with the energy guard,
# HLLD with GLM cleaning, SSP Runge-Kutta), term by term in the order the
# reference program evaluates it: its limiters are switches, so another order
# of summation would grow into a different flow.

def _axis(lo, hi, n, gravity):
    """Cell centres, faces and inverse widths with two ghosts: running sums."""
    dxi = np.full(n + 4, (hi - lo) / float(n))
    dx = dxi.copy()
    dx[1:] = 0.5 * (dxi[:-1] + dxi[1:])
    x, xi = np.zeros(n + 4), np.zeros(n + 4)
    x[1], xi[1] = lo - dxi[1] * 0.5, lo
    x[0], xi[0] = x[1] - dx[1], lo - dxi[1]
    for q in range(2, n + 4):
        x[q], xi[q] = x[q - 1] + dx[q], xi[q - 1] + dxi[q]
    return {"x": x, "xi": xi, "dx": dxi if gravity else dx, "dxi": dxi}


def _min(a, b):
    return torch.where(a < b, a, b)


def _max(a, b):
    return torch.where(a > b, a, b)


def _sgn(a, b):
    return torch.copysign(torch.full_like(b, a), b)


class _Plain:
    def __init__(self, case, n, seed):
        self.case, self.prm, self.n = case, _params(case, n), n
        prm = self.prm
        f = _fields(case, n, prm, seed)
        self.dev, self.gam, self.mag = f["d"].device, prm.gamma, prm.mag_on
        self.grav = prm.gravswitch == 3
        self.dirs = [a for a in range(3) if n[a] > 1]
        self.free = prm.bc[0] == 3
        self.ax = []
        for a in range(3):
            t = {}
            for k, h in _axis(prm.lo[a], prm.hi[a], n[a], self.grav).items():
                t[k] = torch.from_numpy(h).to(self.dev).reshape(
                    [-1 if 2 - a == q else 1 for q in range(3)])
            t["idx"], t["idxi"] = 1.0 / t["dx"], 1.0 / t["dxi"]
            self.ax.append(t)
        d, v, b = f["d"], f["v"], f["b"]
        e = (f["p"] / (self.gam - 1.0) + (d * 0.5) * ((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2])) \
            + 0.5 * ((b[0] * b[0] + b[1] * b[1]) + b[2] * b[2])
        self.glm = self.mag and len(self.dirs) > 1
        self.d, self.v, self.e, self.b = d, list(v), e, list(b)
        self.phi = torch.zeros_like(d)
        self.u = [d, d * v[0], d * v[1], d * v[2], e] + (list(b) if self.mag else []) \
            + ([self.phi] if self.glm else [])
        self.spc = list(f.get("spc", ()))
        self.eint = self.get_eint(e, d, self.v, self.b)
        self.time, self.grvtime, self.cg_old = 0.0, 0.0, 0.0
        if self.grav:
            self.gphi = f["grvphi"][1:-1, 1:-1, 1:-1].clone()
            self.gpsi = torch.zeros_like(d)

    def get_eint(self, e, d, v, b):
        out = e - 0.5 * d * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2])
        if self.mag:
            out = out - 0.5 * (b[0] * b[0] + b[1] * b[1] + b[2] * b[2])
        return out

    @staticmethod
    def fast(d, cs, b1, b2, b3):
        asq, bb1 = cs * cs, b1 * b1 / d
        s = asq + (bb1 + b2 * b2 / d + b3 * b3 / d)
        return torch.sqrt(0.5 * (s + torch.sqrt(s * s - 4.0 * asq * bb1)))

    def cut(self, t, a, lo, count):
        return t.narrow(2 - a, lo, count)

    def coord(self, a, key, lo, count):
        return self.ax[a][key].narrow(2 - a, lo, count)

    def ghosts(self, q, a):
        n, ax = self.n[a], 2 - a
        if self.free:
            lo, hi = self.cut(q, a, 0, 1), self.cut(q, a, n - 1, 1)
            return torch.cat([lo, lo, q, hi, hi], ax)
        return torch.cat([self.cut(q, a, n - 2, 2), q, self.cut(q, a, 0, 2)], ax)

    def slope(self, q, a, m):
        """Limited slope of the m cells -1 .. n."""
        ul, u, ur = (self.cut(q, a, s, m) for s in (0, 1, 2))
        lim = self.case["limiter"]
        if lim == "flat":
            return torch.zeros_like(u)
        if lim == "minmod":
            ia, ib = self.coord(a, "idx", 1, m), self.coord(a, "idx", 2, m)
            x, y = 1.4 * (ur - u) * ib, 1.4 * (u - ul) * ia
            z = (ur - ul) * ia * ib / (ia + ib)
            s = _sgn(1.0, x)
            return s * _max(torch.zeros_like(x), _min(_min(x.abs(), s * y), s * z))
        xm, x0, xp = (self.coord(a, "x", s, m) for s in (0, 1, 2))
        xim, xi0 = self.coord(a, "xi", 0, m), self.coord(a, "xi", 1, m)
        top = (u - ul) * (xp - x0) / (x0 - xm)
        bot = ur - u
        s = _sgn(1.0, bot)
        cf, cb = (xp - x0) / (xi0 - x0), (x0 - xm) / (x0 - xim)
        return s * _max(torch.zeros_like(s), _min(_min(s * 0.5 * (bot + top), s * cf * bot),
                                                  s * cb * top)) / (xp - x0)

    def flux(self, a, ch):
        """(divergence of every conserved variable, of every species)."""
        n, m, gam = self.n[a], self.n[a] + 2, self.gam
        g1 = [self.ghosts(t, a) for t in [self.d, self.e, *self.v, *self.b, self.phi, self.eint]]
        d, w, b = g1[0], g1[2:5], g1[5:8]
        # ghost energies from the ghost pressure
        gm1 = torch.full_like(d, gam - 1.0)
        ge = gm1 * g1[9] / gm1
        gt = ge + 0.5 * (d * (w[0] * w[0] + w[1] * w[1] + w[2] * w[2])
                         + b[0] * b[0] + b[1] * b[1] + b[2] * b[2])
        for k, inner, ghost in ((9, self.eint, ge), (1, self.e, gt)):
            g1[k] = torch.cat([self.cut(ghost, a, 0, 2), inner, self.cut(ghost, a, n + 2, 2)], 2 - a)
        qs = [d, g1[1], d * g1[2], d * g1[3], d * g1[4], g1[5], g1[6], g1[7]]
        phi, ei = g1[8], g1[9]
        if not self.mag:
            qs = qs[:5]
        x0 = self.coord(a, "x", 1, m)
        hl, hr = x0 - self.coord(a, "xi", 0, m), self.coord(a, "xi", 1, m) - x0
        S = [self.slope(q, a, m) for q in qs]
        c = [self.cut(q, a, 1, m) for q in qs]
        fl, fr = [q - hl * s for q, s in zip(c, S)], [q + hr * s for q, s in zip(c, S)]
        bad = torch.zeros_like(c[0], dtype=torch.bool)
        em = self.cut(ei, a, 1, m)
        for w, nb in ((fl, 0), (fr, 2)):
            k = w[1] - 0.5 * (w[2] * w[2] + w[3] * w[3] + w[4] * w[4]) / w[0]
            if self.mag:
                k = k - 0.5 * (w[5] * w[5] + w[6] * w[6] + w[7] * w[7])
            other = self.cut(ei, a, nb, m)
            lo, hi = (other, em) if nb == 0 else (em, other)
            bad = bad | (k >= _max(lo, hi)) | (k <= _min(lo, hi))
        S = [torch.where(bad, torch.zeros_like(s), s) for s in S]
        k = n + 1  # faces -1 .. n-1
        dx1 = self.coord(a, "xi", 1, k) - self.coord(a, "x", 1, k)
        dx2 = self.coord(a, "x", 2, k) - self.coord(a, "xi", 1, k)
        L = [self.cut(q, a, 0, k) + dx1 * self.cut(s, a, 0, k) for q, s in zip(c, S)]
        R = [self.cut(q, a, 1, k) - dx2 * self.cut(s, a, 1, k) for q, s in zip(c, S)]
        rot = [a, (a + 1) % 3, (a + 2) % 3]
        zero = torch.zeros_like(L[0])

        def side(F):
            dd, e = F[0], F[1]
            v = [F[2 + q] / dd for q in rot]
            b = [F[5 + q] for q in rot] if self.mag else [zero] * 3
            pt = (gam - 1.0) * self.get_eint(e, dd, v, b)
            cs = torch.sqrt(gam * pt / dd)
            if self.mag:
                pt = pt + 0.5 * (b[0] * b[0] + b[1] * b[1] + b[2] * b[2])
            return dd, e, v, b, pt, self.fast(dd, cs, *b)
        pl, pr = self.cut(phi, a, 1, k), self.cut(phi, a, 2, k)
        t = self.hlld(side(L), side(R), pl, pr, ch)
        ix = self.coord(a, "idxi", 2, n)

        def div(f):
            return ix * (self.cut(f, a, 0, n) - self.cut(f, a, 1, n))
        out = [None] * 9
        out[0], out[4], out[8] = div(t[0]), div(t[4]), div(t[8])
        for q in range(3):
            out[1 + rot[q]], out[5 + rot[q]] = div(t[1 + q]), div(t[5 + q])
        sp = []
        if self.spc:
            full = [self.ghosts(s, a) for s in self.spc]
            sl = [self.slope(s, a, m) for s in full]
            l_ = [self.cut(s, a, 1, k) + dx1 * self.cut(w, a, 0, k) for s, w in zip(full, sl)]
            r_ = [self.cut(s, a, 2, k) - dx2 * self.cut(w, a, 1, k) for s, w in zip(full, sl)]
            sg = _sgn(0.5, t[0])
            fix = 1.0 / (sum(l_[1:], l_[0]) * (0.5 + sg) + sum(r_[1:], r_[0]) * (0.5 - sg))
            sp = [div(fix * t[0] * (x * (0.5 + sg) + y * (0.5 - sg))) for x, y in zip(l_, r_)]
        return out[:len(self.u)], sp

    @staticmethod
    def hlld(L, R, phil, phir, ch):
        dl, el, (ul, vl, wl), (bl, bl2, bl3), pl, cl = L
        dr, er, (ur, vr, wr), (br, br2, br3), pr, cr = R
        zero = torch.zeros_like(dl)
        b1 = 0.5 * ((bl + br) - (phir - phil) / ch)
        phi = 0.5 * ((phil + phir) - (br - bl) * ch)
        sl, sr = _min(_min(ur - cr, ul - cl), zero), _max(_max(ur + cr, ul + cl), zero)
        av, bv = sl - ul, sr - ur
        den = bv * dr - av * dl
        sm = (bv * dr * ur - av * dl * ul - pr + pl) / den
        pt = (bv * dr * pl - av * dl * pr + dl * dr * bv * av * (ur - ul)) / den

        def star(s, d, e, u, v, w, c2, c3, p, k):
            m = s - sm
            ds = d * k / m
            q = d * k * m - b1 * b1
            v2, v3 = v - b1 * c2 * (sm - u) / q, w - b1 * c3 * (sm - u) / q
            num = d * k * k - b1 * b1
            b2, b3 = c2 * num / q, c3 * num / q
            es = (k * e - p * u + pt * sm + b1 * ((u * b1 + v * c2 + w * c3)
                                                 - (sm * b1 + v2 * b2 + v3 * b3))) / m
            return ds, torch.sqrt(ds), v2, v3, b2, b3, es
        dla, ql, v2l, v3l, b2l, b3l, ela = star(sl, dl, el, ul, vl, wl, bl2, bl3, pl, av)
        dra, qr, v2r, v3r, b2r, b3r, era = star(sr, dr, er, ur, vr, wr, br2, br3, pr, bv)
        sla, sra = sm - b1.abs() / ql, sm + b1.abs() / qr
        s1, qq, qp = _sgn(1.0, b1), ql + qr, torch.sqrt(dla * dra)
        v2a = (ql * v2l + qr * v2r + (b2r - b2l) * s1) / qq
        v3a = (ql * v3l + qr * v3r + (b3r - b3l) * s1) / qq
        b2a = (ql * b2r + qr * b2l + qp * (v2r - v2l) * s1) / qq
        b3a = (ql * b3r + qr * b3l + qp * (v3r - v3l) * s1) / qq
        vb = v2a * b2a + v3a * b3a
        era2 = era + s1 * qr * ((v2r * b2r + v3r * b3r) - vb)
        ela2 = ela - s1 * ql * ((v2l * b2l + v3l * b3l) - vb)
        h, sg = 0.5, _sgn(0.5, sm)
        wl_, wr_, wa = h + _sgn(h, sla), h + _sgn(h, -sra), h - _sgn(h, sla * sra)
        d_ = (h + sg) * dla + (h - sg) * dra
        v2, v3 = wl_ * v2l + wa * v2a + wr_ * v2r, wl_ * v3l + wa * v3a + wr_ * v3r
        b2, b3 = wl_ * b2l + wa * b2a + wr_ * b2r, wl_ * b3l + wa * b3a + wr_ * b3r
        e_ = wl_ * ela + (h - _sgn(h, sla * sm)) * ela2 + (h + _sgn(h, -sm * sra)) * era2 \
            + (h - _sgn(h, sra)) * era
        return [d_ * sm, d_ * sm * sm + pt - b1 * b1, d_ * sm * v2 - b1 * b2,
                d_ * sm * v3 - b1 * b3,
                (e_ + pt) * sm - b1 * (sm * b1 + v2 * b2 + v3 * b3), phi, b2 * sm - b1 * v2,
                b3 * sm - b1 * v3, ch * ch * b1]

    def widths(self):
        return [self.coord(a, "dxi", 2, self.n[a]) for a in range(3)]

    def timestep(self):
        cs = torch.sqrt(self.gam * ((self.gam - 1.0) * self.eint) / self.d)
        x = self.widths()
        den, top = 0.0, None
        b = self.b
        for a in range(3):
            o = [b[a]] + [b[q] for q in range(3) if q != a]
            cf = (self.fast(self.d, cs, *o) if self.mag else cs) + self.v[a].abs()
            area = x[(a + 1) % 3] * x[(a + 2) % 3] if a != 1 else x[0] * x[2]
            den = den + cf * (1.0 if a in self.dirs else 0.0) * (area + area)
            top = cf if top is None else _max(top, cf)
        return self.prm.courant * float((x[0] * x[1] * x[2] / den).min()), top.max()

    def lap(self, ph):
        x = self.widths()
        ia = [self.coord(a, "idx", 2, self.n[a]) for a in range(3)]
        ib = [self.coord(a, "idx", 3, self.n[a]) for a in range(3)]
        area = [x[1] * x[2], x[0] * x[2], x[0] * x[1]]

        def at(a, s):
            o = [1, 1, 1]
            o[a] += s
            return ph[o[2]:o[2] + self.n[2], o[1]:o[1] + self.n[1], o[0]:o[0] + self.n[0]]
        c0 = -((ia[0] + ib[0]) * x[1] * x[2] + (ia[1] + ib[1]) * x[0] * x[2]
               + (ia[2] + ib[2]) * x[0] * x[1])
        out = c0 * at(0, 0)
        for a in self.dirs:
            out = out + area[a] * ia[a] * at(a, -1)
            out = out + area[a] * ib[a] * at(a, 1)
        return out / (x[0] * x[1] * x[2])

    def gravity(self, dt, ch):
        prm, x = self.prm, [float(self.ax[a]["dxi"].flatten()[2]) for a in range(3)]
        sa = [x[1] * x[2], x[0] * x[2], x[0] * x[1]]
        unit = x[0] * x[1] * x[2] / sum((sa[a] + sa[a]) for a in self.dirs)
        cg = prm.HGfac * ch
        dtg = min(prm.hgcfl * unit / cg, dt)
        sub = math.ceil((self.time + dt - self.grvtime) / dtg)
        dtg = (self.time + dt - self.grvtime) / float(sub)
        src = 4.0 * math.acos(-1.0) * prm.G * self.d
        for _ in range(sub):
            damp = math.exp(-(1.0 - self.cg_old / cg + prm.alphagrv * prm.hgcfl))
            p, q = self.gphi[1:-1, 1:-1, 1:-1].clone(), self.gpsi
            p1 = 1.0 * p + 0.0 * p + 1.0 * dtg * cg * q
            q1 = 1.0 * q + 0.0 * q + 1.0 * dtg * cg * (self.lap(self.gphi) - src)
            self.gphi[1:-1, 1:-1, 1:-1] = p1
            q2 = 0.5 * q + 0.5 * q1 + 0.5 * dtg * cg * (self.lap(self.gphi) - src)
            self.gphi[1:-1, 1:-1, 1:-1] = 0.5 * p + 0.5 * p1 + 0.5 * dtg * cg * q1
            self.gpsi = q2 * damp
            self.grvtime, self.cg_old = self.grvtime + dtg, cg

    def source(self):
        ph, out = self.gphi, []
        for a in range(3):
            n = self.n[a]
            dx, dxp = self.coord(a, "dx", 2, n), self.coord(a, "dx", 3, n)
            ix, ixp = self.coord(a, "idx", 2, n), self.coord(a, "idx", 3, n)

            def at(s):
                o = [1, 1, 1]
                o[a] += s
                return ph[o[2]:o[2] + self.n[2], o[1]:o[1] + self.n[1], o[0]:o[0] + self.n[0]]
            out.append(-((dx * ixp * at(1) - dxp * ix * at(-1)) / (dx + dxp)
                         + (dxp - dx) * ix * ixp * at(0)) * self.d)
        return out + [out[0] * self.v[0] + out[1] * self.v[1] + out[2] * self.v[2]]

    def step(self, tn):
        dt, ch = self.timestep()
        if self.grav and tn > 0:
            self.gravity(dt, float(ch))
        u0, s0 = list(self.u), [s * self.d for s in self.spc]
        table = {3: ((1.0, 1.0, 0.0), (0.75, 0.25, 0.25), (1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0)),
                 2: ((1.0, 1.0, 0.0), (0.5, 0.5, 0.5))}[self.case["rk"]]
        for fo, ft, fn in table:
            src = self.source() if self.grav else None
            acc, asp = None, None
            for a in range(3):
                if a in self.dirs:
                    du, sp = self.flux(a, ch)
                else:
                    du, sp = [torch.zeros_like(self.d)] * len(self.u), \
                        [torch.zeros_like(self.d)] * len(self.spc)
                acc = du if acc is None else [p + q for p, q in zip(acc, du)]
                asp = sp if asp is None else [p + q for p, q in zip(asp, sp)]
            if src is not None:
                acc = [q + (src[k - 1] if 1 <= k <= 4 else 0.0) for k, q in enumerate(acc)]
            old = self.d
            self.u = [fo * p + fn * q + ft * dt * r for p, q, r in zip(u0, self.u, acc)]
            self.spc = [(fo * p + fn * q * old + ft * dt * r) / self.u[0]
                        for p, q, r in zip(s0, self.spc, asp)]
            self.d, self.e = self.u[0], self.u[4]
            self.v = [self.u[1 + q] / self.d for q in range(3)]
            if self.mag:
                self.b = self.u[5:8]
            if self.glm:
                self.phi = self.u[8]
            self.eint = self.get_eint(self.e, self.d, self.v, self.b)
        if self.glm:
            self.phi = self.phi * math.exp(-self.prm.alpha9wave * self.prm.courant)
        self.time += dt

    def answer(self, tn):
        def padded(a):
            h = np.zeros([s + 4 for s in self.d.shape])
            h[2:-2, 2:-2, 2:-2] = a.cpu().numpy()
            return h
        out = [self.d, *self.v, self.e] + ([*self.b, self.phi] if self.mag else []) + self.spc
        if self.grav:
            out += [self.gphi[1:-1, 1:-1, 1:-1], self.gpsi]
        fields = [padded(t) for t in out]
        if self.case["loop"] == "batch":
            fields = np.stack(fields)
        elif self.mag and self.case["precision"] == "fp32mix":
            fields[8] = None  # the cleaning field is at that solver's rounding level
        return {"time": self.time, "tn": tn, "fields": fields}


def exact(case, seed):
    sizes = _sizes(case)
    cells = sum(a * b * c for a, b, c in sizes)
    dims = sum(sum(x > 1 for x in n) for n in sizes)
    # seconds: about 350 operations per direction and stage, 10 us each plus
    # their share of memory traffic
    if case["steps"] * case["rk"] * 350 * (1e-5 * dims + 1.6e-11 * cells) > 15.0:
        return None
    out = []
    for q, n in enumerate(sizes):
        p = _Plain(case, n, seed + 1000 * q)
        for tn in range(case["steps"]):
            p.step(tn)
        out.append(p.answer(case["steps"]))
    return out
