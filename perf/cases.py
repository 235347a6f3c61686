"""Workloads for timing the polar-grid particle-mesh framework.

Each case is one call pattern of a program that uses the library, at a size
such a program uses it with:

  run       galaxy's loop: a 2-D disc advanced `steps` steps from its present
            state, then the particles copied back (a snapshot)
  run3      the same on the 3-D grid
  ensemble  independent 2-D discs advanced together, then copied back
  start     particles loaded from host arrays, assigned, the field solved, the
            velocities time-centred, everything copied back (what writing a
            dump's start state needs)
  analysis  the potential solve, the global integrals and the log-spiral
            coefficients of a disc held on the GPU, and its field
  gradient  |A_2|^2 after `steps` steps differentiated in every initial
            velocity, Toomre Q and the disc mass

The discs are exponential discs in a rigid halo (galaxy_amd/disc.py), drawn
here on the GPU.  exact() restates the step in FP64 torch: CIC or quadratic
weights, convolution with the softened point-mass kernels by plain FFTs, the
leap-frog with time-step zones.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from galaxy_amd import adjoint, configs
from galaxy_amd.lib15 import P2DEnsemble, P2DGrid, P3DGrid

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
ZBR = (0.0, 1.5, 3.5)          # zone boundaries, disc scale lengths
NSTEP = (1, 2, 4)
EPS, MD, RTRUNC, RCORE, REDGE, Z0 = 0.1, 0.5, 5.0, 0.1, 6.0, 0.1


def listed():
    run = dict(kind="run", sectors=1, zones=1, fp64=False, comp=False, sort=20)
    run3 = dict(kind="run3", jmass=2, zones=1, fp64=False, sort=8)
    return [
        # a bar-mode test of the size of the reference's own example: one
        # even harmonic, two sectors, two zones, few particles; launch-bound
        dict(run, name="run_small", nr=93, na=128, hash=2, sectors=2, zones=2, n=25_000,
             steps=100),
        # the plain method: FP64, 128 x 128, 1e5 particles
        dict(run, name="run_plain_fp64", nr=128, na=128, hash=8, n=100_000, steps=100,
             fp64=True),
        # the headline size: 256 x 512, 1e7 particles, three zones
        dict(run, name="run_zones", nr=256, na=512, hash=16, zones=3, n=10_000_000, steps=500),
        # the same grid in FP64, an odd particle count
        dict(run, name="run_zones_fp64", nr=256, na=512, hash=16, zones=3, n=3_000_017,
             steps=120, fp64=True),
        # a long integration's option: compensated positions, a grid that is
        # no power of two
        dict(run, name="run_compensated", nr=150, na=300, hash=12, n=2_000_003, steps=120,
             comp=True),
        # a survey of models: 64 discs of uneven size in one context, steps
        # replayed as graphs, the contraction on the matrix cores
        dict(kind="ensemble", name="ensemble", nmem=64, nr=128, na=256, hash=8, nmin=10_000,
             nmax=400_000, steps=120, mfma=True, graph=True, fp64=False, sort=20),
        # a thick disc on the 3-D grid
        dict(run3, name="run3_linear", nr=200, na=256, ngz=125, hash=8, n=20_000_000, steps=100),
        # 3-D with the smoother interpolation, FP64, two zones, a small ragged grid
        dict(run3, name="run3_quadratic_fp64", nr=61, na=90, ngz=45, hash=6, n=600_011, steps=40,
             jmass=3, zones=2, fp64=True),
        # a start state from particle files
        dict(kind="start", name="start", nr=128, na=256, hash=8, zones=3, n=4_000_000,
             fp64=False),
        # what a run does at its analysis steps
        dict(kind="analysis", name="analysis", nr=256, na=512, hash=16, zones=3, n=10_000_000,
             fp64=False, pitches=25, harmonics=6),
        # the differentiated run, and a small one in FP64
        dict(kind="gradient", name="gradient", nr=128, na=256, hash=8, n=1_000_000, steps=100,
             every=20, fp64=False),
        dict(kind="gradient", name="gradient_small_fp64", nr=96, na=128, hash=4, n=20_000,
             steps=40, every=10, fp64=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, c, na_lo, na_hi):
    c["na"] = 2 * _log(rng, na_lo // 2, na_hi // 2)
    c["nr"] = max(40, int(c["na"] * rng.uniform(0.5, 0.9)))
    c["hash"] = rng.choice((2, 4, 6, 8, 11, 16))
    return c


def draw(rng):
    kind = rng.choice(("run", "run", "run", "run3", "ensemble", "start", "analysis", "gradient"))
    c = dict(kind=kind, fp64=rng.random() < 0.35)
    if kind == "run":
        _grid(rng, c, 90, 512)
        c.update(sectors=rng.choice((1, 1, 2)), zones=rng.choice((1, 2, 3)), comp=False,
                 n=_log(rng, 5_000, 6_000_000), steps=rng.randint(40, 120),
                 sort=rng.choice((10, 16, 20)))
        c["comp"] = not c["fp64"] and rng.random() < 0.3
    elif kind == "run3":
        _grid(rng, c, 90, 256)
        c.update(ngz=rng.randint(31, 125), hash=rng.choice((2, 4, 6, 8)), jmass=rng.choice((2, 2, 3)),
                 zones=rng.choice((1, 2)), n=_log(rng, 100_000, 8_000_000),
                 steps=rng.randint(16, 40), sort=rng.choice((5, 8)))
        if c["fp64"]:
            c["n"], c["ngz"], c["hash"] = c["n"] // 4, min(c["ngz"], 61), min(c["hash"], 6)
    elif kind == "ensemble":
        _grid(rng, c, 90, 256)
        c.update(nmem=rng.randint(3, 64), hash=rng.choice((4, 8)), nmin=5_000,
                 nmax=_log(rng, 20_000, 300_000), steps=rng.randint(40, 120),
                 graph=rng.random() < 0.5, sort=rng.choice((10, 20)))
        c["mfma"] = not c["fp64"] and rng.random() < 0.5
    elif kind == "start":
        _grid(rng, c, 90, 512)
        c.update(zones=rng.choice((1, 2, 3)), n=_log(rng, 10_000, 4_000_000))
    elif kind == "analysis":
        _grid(rng, c, 90, 512)
        c.update(zones=rng.choice((1, 2, 3)), n=_log(rng, 10_000, 10_000_000),
                 pitches=rng.choice((9, 25, 41)), harmonics=rng.randint(1, 8))
    else:
        _grid(rng, c, 90, 256)
        c.update(hash=rng.choice((2, 4, 8)), n=_log(rng, 10_000, 1_000_000),
                 steps=rng.randint(20, 80), every=rng.choice((10, 20)))
    return c


# ---- models --------------------------------------------------------------------


def _workload(c, n):
    """The case's disc as a workload of galaxy_amd.configs."""
    nz = c.get("zones", 1)
    kw = dict(name="case", nr=c["nr"], na=c["na"], hash=c["hash"], n=n,
              steps=c.get("steps", 1), dt=0.025 if nz > 1 else 0.05, nstep=NSTEP[:nz],
              zbr_model=ZBR[:nz], eps_model=EPS, md=MD, rtrunc=RTRUNC, rcore=RCORE, redge=REDGE)
    if "ngz" in c:
        # the planes reach fifteen scale heights either side of the mid-plane,
        # their spacing below the softening length
        return configs.Workload3(ngz=c["ngz"], dz_model=min(0.09, 31 * Z0 / (c["ngz"] - 1)),
                                 z0=Z0, **kw)
    return configs.Workload(**kw)


def _particles(w, n, seed, Q, fp64):
    """One disc's particles in internal units as host arrays of the run's
    precision: x, y[, z], vx, vy[, vz], zones."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    u = torch.rand(n, generator=g, device=DEV, dtype=F64)
    phi = torch.rand(n, generator=g, device=DEV, dtype=F64) * (2 * math.pi)
    gR, gp = (torch.randn(n, generator=g, device=DEV, dtype=F64) for _ in range(2))
    mt = 1.0 - (1.0 + RTRUNC) * math.exp(-RTRUNC)
    tgt = u * mt
    R = torch.where(tgt < 0.5, torch.sqrt(2 * tgt), 2 - torch.log1p(-tgt)).clamp(0, RTRUNC)
    for _ in range(8):
        f = 1 - (1 + R) * torch.exp(-R) - tgt
        R = (R - f / (R * torch.exp(-R)).clamp_min(1e-300)).clamp(0, RTRUNC)
    s2 = R * R + RCORE ** 2
    kap2 = 2 * (R * R + 2 * RCORE ** 2) / (s2 * s2)
    sig = w.md / (2 * math.pi * mt) * torch.exp(-R)
    sR = 3.36 * Q * sig / torch.sqrt(kap2)
    k4 = kap2 * s2 / 4                       # kappa^2 / (4 Omega^2)
    # d ln(Sigma sigma_R^2) / d ln R
    dlog = -3 * R - 2 * R * R / (R * R + 2 * RCORE ** 2) + 4 * R * R / s2
    vm = torch.sqrt((R * R / s2 + sR * sR * (dlog + 1 - k4)).clamp_min(0))
    vR, vp = sR * gR, vm + sR * torch.sqrt(k4) * gp
    ls, ts = w.lscale(), w.dt
    cp, sp = torch.cos(phi), torch.sin(phi)
    pos = [R * cp * ls, R * sp * ls]
    vel = [(vR * cp - vp * sp) * ls * ts, (vR * sp + vp * cp) * ls * ts]
    r = R * ls
    off = r > w.rgrid_d()
    if isinstance(w, configs.Workload3):
        v = torch.rand(n, generator=g, device=DEV, dtype=F64)
        z = Z0 * torch.atanh((2 * v - 1).clamp(-1 + 1e-15, 1 - 1e-15))
        gz = torch.randn(n, generator=g, device=DEV, dtype=F64)
        pos.append(z * ls)
        vel.append(torch.sqrt(math.pi * sig * Z0) * gz * ls * ts)
        r = torch.sqrt(R * R + z * z) * ls
        off |= pos[2].abs() > configs.zmax3(w)
    iz = torch.ones(n, dtype=torch.int32, device=DEV)
    for i in range(1, w.nzones):
        iz[r >= ZBR[i] * ls] = i + 1
    fac = torch.tensor(w.nstep, dtype=F64, device=DEV)[iz.long() - 1]
    iz[off] = w.nzones + 1
    dt = F64 if fp64 else torch.float32
    return [a.to(dt).cpu().numpy() for a in pos + [v * fac for v in vel]] + [iz.cpu().numpy()]


def _precision(c):
    return "fp64" if c["fp64"] else "fp32"


def _grid_args(c, w):
    kw = configs.grid_kwargs3(w) if "ngz" in c else configs.grid_kwargs(w)
    kw["nsect"] = c.get("sectors", 1)
    kw["offanal"] = True
    if "jmass" in c:
        kw["jmass"] = c["jmass"]
    return kw


def _rmax(g):
    return math.sqrt(g.rgrid ** 2 + g.zm ** 2) if isinstance(g, P3DGrid) else g.rgrid


def _members(c):
    """The members' sizes (log-uniform) and Toomre Q, fixed by the case."""
    rng = np.random.default_rng(4)
    counts = np.exp(rng.uniform(math.log(c["nmin"]), math.log(c["nmax"]), c["nmem"])).astype(int)
    return [int(k) for k in counts], [float(q) for q in rng.uniform(1.0, 2.0, c["nmem"])]


def _member_particles(c, seed):
    counts, Q = _members(c)
    return [_particles(_workload(c, k), k, seed * 1000 + i, Q[i], c["fp64"])
            for i, k in enumerate(counts)]


def _set_tables(g, w):
    g.greenm()
    g.set_fixforce(*configs.fixforce(w, _rmax(g)))
    g.set_fixpot(*configs.fixpot(w, _rmax(g)))


def prepare(case, seed):
    c = case
    if c["kind"] == "gradient":
        w = _workload(c, c["n"])
        w.Q, w.seed = 1.2, seed
        return c, adjoint.DiscModel(w, precision=_precision(c))
    if c["kind"] == "ensemble":
        counts, _ = _members(c)
        w = _workload(c, 1)
        kw = _grid_args(c, w)
        kw["pmass"] = [kw["pmass"] / k for k in counts]
        g = P2DEnsemble(c["nmem"], precision=_precision(c), **kw)
        if c["mfma"]:
            g.set_contraction("mfma", 0)
        _set_tables(g, w)
        g.restrt(_member_particles(c, seed))
        g.masset()
        g.set_sort_interval(c["sort"])
        g.set_graph(c["graph"])
        return c, g
    w = _workload(c, c["n"])
    cls = P3DGrid if "ngz" in c else P2DGrid
    g = cls(precision=_precision(c), **_grid_args(c, w))
    if c.get("comp"):
        g.set_compensated(True)
    _set_tables(g, w)
    p = _particles(w, c["n"], seed, 1.5, c["fp64"])
    if c["kind"] == "start":
        return c, g, p
    g.restrt(*p)
    g.masset()
    if c["kind"] == "analysis":
        return c, g, w.lscale()
    g.set_sort_interval(c["sort"])
    return c, g


def run(state):
    c, g = state[:2]
    if c["kind"] == "gradient":
        r = g.gradient(1.2, MD, c["steps"], every=c["every"])
        return {k: r[k] for k in ("loss", "dvx", "dvy", "dQ", "dmd", "gpar")}
    if c["kind"] == "start":
        g.set_step(0)
        g.restrt(*state[2])
        g.masset()
        g.findf(True)
        g.tmcent(True)
        mass, _, jrad, krad, _ = g.get_mass()
        return {"particles": g.unload(), "field": g.get_field(), "mass": mass, "jrad": jrad,
                "krad": krad}
    if c["kind"] == "analysis":
        g.findf(True)
        return {"integrals": g.integrals(),
                "spirals": g.lgspia(c["pitches"], c["harmonics"], state[2]),
                "field": g.get_field()}
    g.run(c["steps"])
    if c["kind"] == "ensemble":
        # unload's members are slices of one array each; the whole arrays
        first = g.unload()[0]
        return {k: v.base for k, v in first.items()}
    out = g.unload()
    if c.get("comp"):
        out["xlo"], out["ylo"] = g.get_position_lo()
    return out


# ---- what a pass cannot do without -----------------------------------------------


def _pushes(c):
    """Pushes of one step per particle: zone i's share of the disc / nstep_i."""
    nz = c.get("zones", 1)
    m = [1 - (1 + r) * math.exp(-r) for r in ZBR[:nz] + (RTRUNC,)]
    return sum((m[i + 1] - m[i]) / m[nz] / NSTEP[i] for i in range(nz))


def work(case):
    c = case
    es = 8 if c["fp64"] else 4
    nm = 1
    n = c.get("n")
    if c["kind"] == "ensemble":
        nm = c["nmem"]
        lo, hi = math.log(c["nmin"]), math.log(c["nmax"])
        n = int(nm * (c["nmax"] - c["nmin"]) / (hi - lo))
    d3 = "ngz" in c
    ng = c["hash"] // c.get("sectors", 1) + 1
    mesh = c["nr"] * c["na"] * c.get("ngz", 1)
    nw = 4 if not d3 else 8 if c["jmass"] == 2 else 27
    comps = 3 if d3 else 2
    state = 2 * comps * es                             # position and velocity
    snap = n * (state + 4)                             # a copy with the zones
    # tables once; the grids (mass in, field out) once a solve
    table = (comps if d3 else 2) * c.get("ngz", 1) * ng * c["nr"] ** 2 * es
    grids = nm * mesh * es * (1 + comps)
    fft = 5.0 * mesh * math.log2(mesh)                 # one real transform of the mesh
    solve = nm * ((1 + comps) * fft / 2 +
                  comps * c.get("ngz", 1) * ng * 4.0 * c["nr"] ** 2 * (2 if d3 else 1))
    push = 60 + 2 * nw * (comps + 1)                   # operations of one push
    if c["kind"] == "start":
        return {"bytes": 2.0 * snap + table + grids, "flops": solve + n * push}
    if c["kind"] == "analysis":
        return {"bytes": n * (state + 1.0) + table + grids,
                "flops": solve + n * (push + 8.0 * c["pitches"] * c["harmonics"])}
    if c["kind"] == "gradient":
        # forward, then backward with the adjoint read and written
        s = c["steps"]
        return {"bytes": s * (n * (2.0 * state + 2 * 32 + state) + 2 * grids) + table + 2 * snap,
                "flops": s * (n * 3.0 * push + 2 * solve)}
    p = _pushes(c) * n
    return {"bytes": c["steps"] * (p * 2.0 * state + grids) + table + snap,
            "flops": c["steps"] * (p * push + solve)}


# ---- the same in 64 bits -----------------------------------------------------------


class _Exact:
    """The disc's step in FP64 torch: particles, masses, field."""

    def __init__(self, c, w, parts, pmass, rgrid, zm, tables):
        self.c, self.w = c, w
        self.d3 = "ngz" in c
        self.nr, self.na, self.ngz = c["nr"], 2 * (c["na"] // 2), c.get("ngz", 1)
        self.nz, self.nstep = w.nzones, w.nstep
        self.alpha = 2 * math.pi / self.na
        self.rgrid, self.zm, self.pmass = rgrid, zm, pmass
        self.dz = w.dz_model * w.lscale() if self.d3 else 1.0
        self.zbr = [z * w.lscale() for z in w.zbr_model]
        self.sect = c.get("sectors", 1)
        self.mesh = self.nr * self.na * self.ngz
        self.dim = 3 if self.d3 else 2
        up = [torch.as_tensor(a, device=DEV).to(F64) for a in parts[:-1]]
        self.x, self.v = up[:self.dim], up[self.dim:]
        self.iz = torch.as_tensor(parts[-1], device=DEV).long()
        self.force, self.pot = ([torch.as_tensor(t[1], device=DEV), torch.as_tensor(t[2], device=DEV),
                                 float(t[0])] for t in tables)
        self.istep = 0
        self.kernels = {}

    # -- tables and weights
    @staticmethod
    def _table(t, r):
        val, der, dr = t
        n = len(val)
        k = (r / dr).long().clamp(0, n - 2)
        s = r / dr - k
        d0, d1 = dr * der[k], dr * der[k + 1]
        v0, v1 = val[k], val[k + 1]
        c2 = 3 * (v1 - v0) - 2 * d0 - d1
        c3 = 2 * (v0 - v1) + d0 + d1
        return torch.where(r >= dr * (n - 1), val[-1], v0 + s * (d0 + s * (c2 + s * c3)))

    def _corners(self, x, fold):
        """(flat cell index, weight) of each corner of positions x."""
        na = self.na
        u = torch.log1p(torch.hypot(x[0], x[1])) / self.alpha
        t = torch.atan2(x[1], x[0]) / self.alpha
        t = torch.where(t < 0, t + na, t)
        if fold and self.sect > 1:
            t = torch.remainder(t, na / self.sect)
        axes = [(u, self.nr), (t, 0)]
        if self.d3:
            axes.insert(1, ((x[2] + self.zm) / self.dz, self.ngz))
        quad = self.c.get("jmass") == 3
        idx, wts = [], []
        for k, (q, n) in enumerate(axes):
            j = (q + 0.5 * quad).long()
            if n:
                j = j.clamp(1 if quad and k == 0 else 0, n - 2)
            if quad:
                e = q + 0.5 - j
                wts.append([(1 - 2 * e + e * e) / 2, (1 + 2 * e - 2 * e * e) / 2, e * e / 2])
                idx.append([j - 1, j, j + 1])
            else:
                e = q - j
                wts.append([1 - e, e])
                idx.append([j, j + 1])
        for a in range(len(idx[0])):
            for b in range(len(idx[1]) if self.d3 else 1):
                for s in range(len(idx[-1])):
                    cell, wt = idx[0][a], wts[0][a] * wts[-1][s]
                    if self.d3:
                        cell, wt = cell * self.ngz + idx[1][b], wt * wts[1][b]
                    cell = cell * na + torch.remainder(idx[-1][s], na)
                    ok = (cell >= 0) & (cell < self.mesh)
                    yield torch.where(ok, cell, 0), torch.where(ok, wt, 0.0)

    # -- masses
    def _assign(self, sel):
        """Per-zone masses of the particles sel."""
        out = [torch.zeros(self.mesh, dtype=F64, device=DEV) for _ in range(self.nz)]
        for z in range(1, self.nz + 1):
            k = (sel & (self.iz == z)).nonzero().squeeze(1)
            if k.numel():
                for cell, wt in self._corners([a[k] for a in self.x], True):
                    out[z - 1].index_add_(0, cell, wt * self.pmass)
        return out

    def masset(self):
        self.new = self._assign(self.iz <= self.nz)
        self.old = [m.clone() for m in self.new]
        self.due = [0] * self.nz                 # time of the new mass arrays
        self.was = [0] * self.nz

    def density(self):
        rho = self.new[0].clone()
        for z in range(1, self.nz):
            left = self.due[z] - self.istep
            ns = self.nstep[z]
            rho += (1 - left / ns) * self.new[z]
            if left:
                rho += (1 - (self.istep - self.was[z]) / ns) * self.old[z]
        return rho

    # -- the field
    def _kernel(self, kind):
        """Transform of the softened point-mass kernel [k_z, m, field, source]."""
        if kind in self.kernels:
            return self.kernels[kind]
        ng = min(self.c["hash"] + 1, self.na // 2 + 1)
        r = torch.expm1(self.alpha * torch.arange(self.nr, dtype=F64, device=DEV))
        rs, rf = r[None, :, None], r[:, None, None]
        th = self.alpha * torch.arange(self.na, dtype=F64, device=DEV)
        eps = EPS * self.w.lscale()
        base = rs * rs + rf * rf - 2 * rs * rf * torch.cos(th) + eps * eps
        num = {"R": rs * torch.cos(th) - rf, "t": -rs * torch.sin(th)}.get(kind)
        m = torch.arange(ng, dtype=F64, device=DEV)
        keep = (m % self.sect == 0).to(F64)
        ang = torch.polar(torch.ones(1, dtype=F64, device=DEV), -(th[:, None] * m)) * keep
        planes = []
        for k in range(self.ngz + 1 if self.d3 else 1):
            d2 = base + (k * self.dz) ** 2
            f = -1 / torch.sqrt(d2) if kind == "p" else \
                (-k * self.dz if kind == "z" else num) / (d2 * torch.sqrt(d2))
            f = f.expand(self.nr, self.nr, self.na).reshape(-1, self.na)
            planes.append(torch.complex(f @ ang.real.contiguous(), f @ ang.imag.contiguous())
                          .reshape(self.nr, self.nr, ng))
        K = torch.stack(planes)                              # [z, field, source, m]
        if self.d3:
            sign = -1 if kind == "z" else 1
            K[self.ngz] = 0 if kind == "z" else K[self.ngz]
            K = torch.fft.fft(torch.cat([K, sign * K[1:self.ngz].flip(0)]), dim=0)
        self.kernels[kind] = K.permute(0, 3, 1, 2).contiguous()
        return self.kernels[kind]

    def field(self, pot=False):
        """[components, mesh] Cartesian accelerations and, if pot, the potential."""
        ng = min(self.c["hash"] + 1, self.na // 2 + 1)
        rho = self.density().reshape(self.nr, self.ngz, self.na)
        M = torch.fft.rfft(rho, dim=2)[:, :, :ng]
        P = 2 * self.ngz if self.d3 else 1
        if self.d3:
            M = torch.fft.fft(M, n=P, dim=1)
        M = M.permute(1, 2, 0).contiguous()                  # [k_z, m, source]
        F = {}
        for kind in ("R", "t") + (("z",) if self.d3 else ()) + (("p",) if pot else ()):
            K = self._kernel(kind)
            W = torch.stack([(K[k] * M[k][:, None, :]).sum(2) for k in range(P)])
            W = W.permute(2, 0, 1)                           # [field, k_z, m]
            if self.d3:
                W = torch.fft.ifft(W, dim=1)[:, :self.ngz]
            full = torch.zeros(self.nr, self.ngz, self.na // 2 + 1, dtype=torch.complex128,
                               device=DEV)
            full[:, :, :ng] = W
            F[kind] = torch.fft.irfft(full, n=self.na, dim=2)
        th = self.alpha * torch.arange(self.na, dtype=F64, device=DEV)
        co, si = torch.cos(th), torch.sin(th)
        out = [F["R"] * co - F["t"] * si, F["R"] * si + F["t"] * co]
        out += [F[k] for k in ("z", "p") if k in F]
        return torch.stack([f.reshape(-1) for f in out])

    def getacc(self, fld, k):
        """Accelerations of the particles k, zone factor included."""
        x = [a[k] for a in self.x]
        on = (self.iz[k] <= self.nz).to(F64)
        acc = [torch.zeros_like(x[0]) for _ in x]
        for cell, wt in self._corners(x, False):
            for d in range(self.dim):
                acc[d] += wt * fld[d][cell]
        r = torch.sqrt(sum(a * a for a in x))
        f = self._table(self.force, r) / r.clamp_min(1e-300)
        fac = torch.tensor(self.nstep, dtype=F64, device=DEV)[self.iz[k].clamp(max=self.nz) - 1]
        return [(a + f * b) * on * fac * fac for a, b in zip(acc, x)]

    def _zone(self, x):
        r = torch.sqrt(sum(a * a for a in x))
        z = torch.ones_like(r, dtype=torch.long)
        for i in range(1, self.nz):
            z[r >= self.zbr[i]] = i + 1
        return z

    def step(self):
        fld = self.field()
        due = [z for z in range(self.nz) if self.istep % self.nstep[z] == 0]
        mz = max(due) + 1
        nl = self.nz + 1
        k = ((self.iz <= mz) | ((self.iz == nl) & (mz == self.nz))).nonzero().squeeze(1)
        acc = self.getacc(fld, k)
        ns = torch.tensor(self.nstep + (self.nstep[-1],), dtype=F64, device=DEV)
        x, v = [a[k] for a in self.x], [a[k] for a in self.v]
        z0 = self.iz[k]
        new_v = [a + b for a, b in zip(v, acc)]
        new_x = [a + b for a, b in zip(x, new_v)]

        def change(sel, fac):
            for d in range(self.dim):
                ov = fac * (v[d] + 0.5 * acc[d] * (1 - fac))
                na = acc[d] * fac * fac
                v[d], acc[d] = torch.where(sel, ov, v[d]), torch.where(sel, na, acc[d])
                new_v[d] = torch.where(sel, ov + na, new_v[d])
                new_x[d] = torch.where(sel, x[d] + ov + na, new_x[d])

        off = torch.hypot(new_x[0], new_x[1]) > self.rgrid
        if self.d3:
            off |= new_x[2].abs() > self.zm
        was_off = z0 == nl
        z = torch.where(~was_off & off, nl, torch.where(was_off & ~off, self.nz, z0))
        if self.nz > 1:
            change(~was_off & off & (z0 < self.nz), ns[self.nz - 1] / ns[z0 - 1])
        if mz > 1:
            kz = self._zone(new_x).clamp(max=mz)
            kz = torch.where(kz > z, self._zone(x), kz)
            sel = ~was_off & (z <= mz) & (kz != z)
            change(sel, ns[kz - 1] / ns[z - 1])
            z = torch.where(sel, kz, z)
        for d in range(self.dim):
            self.x[d][k], self.v[d][k] = new_x[d], new_v[d]
        self.iz[k] = z
        moved = torch.zeros_like(self.iz, dtype=torch.bool)
        moved[k] = True
        mass = self._assign(moved & (self.iz <= mz))
        for q in range(mz):
            if q:
                self.old[q], self.was[q] = self.new[q], self.due[q]
            self.new[q] = mass[q]
            self.due[q] = self.istep + self.nstep[q]
        self.istep += 1

    def particles(self):
        names = "xyz"[:self.dim]
        return {**dict(zip(names, self.x)), **{"v" + q: a for q, a in zip(names, self.v)},
                "iz": None}


def _exact_disc(c, w, parts, pmass):
    ls = w.lscale()
    alpha = 2 * math.pi / (2 * (c["na"] // 2))
    edge = c["nr"] - (c["jmass"] / 2 if "ngz" in c else 1)
    rgrid = math.exp(alpha * edge) - 1
    zm = 0.5 * w.dz_model * ls * (c["ngz"] + 1 - c["jmass"]) if "ngz" in c else 0.0
    rmax = math.hypot(rgrid, zm)
    return _Exact(c, w, parts, pmass, rgrid, zm,
                  (configs.fixforce(w, rmax), configs.fixpot(w, rmax)))


def _exact_analysis(c, e):
    fld = e.field(True)
    every = torch.arange(c["n"], device=DEV)
    acc = e.getacc(fld, every)
    sf = 1 / torch.tensor(e.nstep, dtype=F64, device=DEV)[e.iz.clamp(max=e.nz) - 1]
    v = [(a + 0.5 * b) * sf for a, b in zip(e.v, acc)]
    pm, on = e.pmass, (e.iz <= e.nz).to(F64)
    phi = sum(wt * fld[2][cell] for cell, wt in e._corners(e.x, False)) * on
    r = torch.hypot(*e.x)
    d = dict(mass=pm * c["n"], cm=torch.stack([a.mean() for a in e.x]),
             momentum=pm * torch.stack([a.sum() for a in v]),
             ke=0.5 * pm * (v[0] ** 2 + v[1] ** 2).sum(),
             lz=pm * (e.x[0] * v[1] - e.x[1] * v[0]).sum(), w_grid=pm * phi.sum(),
             w_fixed=pm * e._table(e.pot, r).sum())
    d["energy"] = d["ke"] + 0.5 * d["w_grid"] + d["w_fixed"]
    th, a = torch.atan2(e.x[1], e.x[0]), 0.25 * torch.log(r / e.w.lscale())
    A = torch.zeros(c["pitches"], c["harmonics"], dtype=torch.complex128, device=DEV)
    for j in range(c["pitches"]):
        for m in range(c["harmonics"]):
            ph = (m + 1) * (th + (j - c["pitches"] // 2) * a)
            A[j, m] = torch.complex(torch.cos(ph).mean(), torch.sin(ph).mean())
    d = {k: float(x) if k not in ("cm", "momentum") else x for k, x in d.items()}
    return {"integrals": d, "spirals": (A.real.reshape(-1), A.imag.reshape(-1)), "field": fld}


def exact(case, seed):
    c = case
    if c["kind"] == "gradient":
        return None       # a reverse sweep in 64 bits would itself be this package's
    if c["kind"] == "ensemble":
        counts, _ = _members(c)
        done = []
        table = None
        for k, parts in zip(counts, _member_particles(c, seed)):
            w = _workload(c, k)
            e = _exact_disc(c, w, parts, configs.grid_kwargs(w)["pmass"])
            e.kernels = table or e.kernels
            e.masset()
            for _ in range(c["steps"]):
                e.step()
            table = e.kernels
            done.append(e.particles())
        return {k: None if k == "iz" else torch.cat([d[k] for d in done]) for k in done[0]}
    w = _workload(c, c["n"])
    parts = _particles(w, c["n"], seed, 1.5, c["fp64"])
    e = _exact_disc(c, w, parts, configs.grid_kwargs(w)["pmass"])
    e.masset()
    if c["kind"] == "analysis":
        return _exact_analysis(c, e)
    if c["kind"] == "start":
        fld = e.field(True)
        acc = e.getacc(fld, torch.arange(c["n"], device=DEV))
        for d in range(e.dim):
            e.v[d] -= 0.5 * acc[d]
        return {"particles": e.particles(), "field": fld, "mass": None, "jrad": None,
                "krad": None}
    for _ in range(c["steps"]):
        e.step()
    out = e.particles()
    if c.get("comp"):
        out["xlo"] = out["ylo"] = None
    return out
