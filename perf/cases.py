"""Timed cases: what programs that use the framework have it do.

A case is a dict of plain values; `listed()` gives the standing ones, `draw()` others of the
same ranges, `prepare()` what a program holds before the call (the scenario on the GPU),
`run()` one pass through the public entry points, `work()` the bytes and operations a pass
cannot do without, `exact()` the outputs of a first pass in 64-bit arithmetic of its own.

Passes (key "use"):
  coupled   a BMI-style coupler: it writes the external sources, takes one step and reads
            the levels
  sweeps    a host that drives the step itself: forcing, momentum, continuity, one call each
  interval  a simulation run from one map output to the next: `span` seconds, then the fields
            the output holds
  ensemble  a batch of scenarios of uneven size advanced together by 32 steps, then the
            levels of each

A pass goes on from where the last one ended, as a running simulation does; forcing repeats
with the tide, so that passes late in a run do the work of early ones.
"""
import math

import numpy as np
import torch

from sfincs_amd import _lib
from sfincs_amd import workloads as W

T_END = 2.0e6         # far beyond what is timed: no pass runs into the end of its scenario
TIDE = 43200.0
SLOPE_LO, SLOPE_HI = -10.0, 5.0


def listed():
    return [
        # a coupled groundwater or sewer model exchanging with a small domain every step
        dict(name="coupled_48x64", use="coupled", mesh="regular", n=48, m=64),
        # a host with its own step loop on a district with subgrid tables
        dict(name="sweeps_subgrid_160x120", use="sweeps", mesh="subgrid", n=160, m=120),
        # a quick look at a small coast: levels, maxima and the flow field every 10 minutes
        dict(name="regular_64x96", use="interval", mesh="regular", n=64, m=96, span=600.0, flow=True, rain=True),
        # a town with subgrid tables on a ragged rectangle
        dict(name="subgrid_161x203", use="interval", mesh="subgrid", n=161, m=203, span=300.0),
        # the 512 x 512 beach of the smallest benchmark workload, under rain
        dict(name="regular_512x512", use="interval", mesh="regular", n=512, m=512, span=300.0, rain=True),
        # a city with rivers
        dict(name="subgrid_512x700", use="interval", mesh="subgrid", n=512, m=700, span=300.0, sources=8),
        # a whole coast at 50 m without subgrid tables, mostly wet
        dict(name="regular_1536x2048", use="interval", mesh="regular", n=1536, m=2048, span=120.0, rain=True),
        # the flagship workload: 2048 x 2048 with subgrid tables and discharges
        dict(name="subgrid_2048x2048", use="interval", mesh="subgrid", n=2048, m=2048, span=120.0, sources=8),
        # quadtree meshes with wind: a harbour, and a coast of 2.6 million cells
        dict(name="quadtree_24", use="interval", mesh="quadtree", n=24, m=24, span=60.0, flow=True),
        dict(name="quadtree_256", use="interval", mesh="quadtree", n=256, m=256, span=30.0),
        # an irregular active area with the slower physics switched on
        dict(name="masked_277x301", use="interval", mesh="masked", n=277, m=301, span=300.0, rain=True),
        # an ensemble of eight regular and subgrid members
        dict(name="ensemble_8", use="ensemble", mesh="mixed", members=8, n=48, m=400),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["coupled", "sweeps", "regular", "regular", "subgrid", "subgrid", "quadtree", "masked", "ensemble"])
    if kind == "coupled":
        return dict(use="coupled", mesh="regular", n=_log(rng, 24, 200), m=_log(rng, 24, 200))
    if kind == "sweeps":
        return dict(use="sweeps", mesh=rng.choice(["regular", "subgrid"]), n=_log(rng, 32, 400), m=_log(rng, 32, 400))
    if kind == "regular":
        return dict(use="interval", mesh="regular", n=_log(rng, 24, 1500), m=_log(rng, 32, 2048), rain=rng.random() < 0.5,
                    span=rng.choice([60.0, 120.0, 300.0]), flow=rng.random() < 0.3)
    if kind == "subgrid":
        return dict(use="interval", mesh="subgrid", n=_log(rng, 32, 1024), m=_log(rng, 32, 1024),
                    span=rng.choice([60.0, 120.0]), sources=rng.choice([0, 3, 8]), flow=rng.random() < 0.3)
    if kind == "quadtree":
        return dict(use="interval", mesh="quadtree", n=_log(rng, 12, 160), m=_log(rng, 12, 160), span=rng.choice([15.0, 30.0]))
    if kind == "masked":
        return dict(use="interval", mesh="masked", n=_log(rng, 32, 600), m=_log(rng, 32, 600), span=rng.choice([60.0, 120.0]),
                    rain=rng.random() < 0.5)
    return dict(use="ensemble", mesh="mixed", members=rng.randint(2, 8), n=_log(rng, 24, 64), m=_log(rng, 80, 400))


# ------------------------------------------------------------------------------- scenarios
def _tide(amp, phase):
    t = np.arange(0.0, T_END + 1200.0, 600.0)
    return t.astype(np.float32), (amp * np.sin(2.0 * np.pi * t / TIDE + phase)).astype(np.float32)[:, None]


def _storms(rate):
    """Two hours of rain in every twelve, from the start on, falling off within ten minutes."""
    t, v = [], []
    for k in range(int(T_END / TIDE) + 2):
        t += [k * TIDE, k * TIDE + 7200.0, k * TIDE + 7800.0, (k + 1) * TIDE - 600.0]
        v += [rate, rate, 0.0, 0.0]
    return np.array(t, np.float32), np.array(v, np.float32)


def _coast(r, n, m, dx):
    """A bed rising from -10 m in the west to +5 m in the east over the whole domain, with
    bumps of up to 2 m: two thirds of it lie below mean sea level."""
    x = (np.arange(m, dtype=np.float32) + 0.5)[:, None] / m
    y = (np.arange(n, dtype=np.float32) + 0.5)[None, :] / n
    zb = SLOPE_LO + (SLOPE_HI - SLOPE_LO) * x + np.zeros_like(y)
    for _ in range(12):
        a, s, px, py = r.uniform(-2.0, 2.0), r.uniform(0.02, 0.1), r.uniform(0.05, 1.0), r.uniform()
        zb = zb + np.float32(a) * (np.exp(-((x - np.float32(px)) / np.float32(s)) ** 2) *
                                   np.exp(-((y - np.float32(py)) / np.float32(s)) ** 2))
    return np.ascontiguousarray(zb, np.float32)


def _regular(case, seed, **params):
    r = W.rng(seed)
    n, m, dx = case["n"], case["m"], 50.0
    zb = _coast(r, n, m, dx)
    msk = np.ones((m, n), np.int8)
    msk[0, :] = 2
    t, zs = _tide(r.uniform(0.5, 1.5), r.uniform(0.0, 1.0))
    sc = W.Scenario(name="regular", params=dict(t0=0.0, t1=T_END, manning=0.02, **params), nmax=n, mmax=m, dx=dx, dy=dx,
                    msk=msk.reshape(-1), zb_grid=zb, t_end=T_END,
                    bnd=(np.array([-dx / 2], np.float32), np.array([n * dx / 2], np.float32), t, zs))
    if case.get("rain"):
        sc.rain = _storms(r.uniform(5.0, 30.0))
    return sc


def _subgrid(case, seed, tables=None):
    """The flagship recipe (fractal terrain, land-use roughness, 10 levels) at any size."""
    n, m = case["n"], case["m"]
    sc = W.subgrid_case(n, m, seed=seed, t_end=7200.0, nsrc=case.get("sources", 0))
    r = W.rng(seed + 1)
    t, zs = _tide(r.uniform(1.0, 2.0), r.uniform(0.0, 1.0))
    x, y = sc.bnd[:2]
    sc.bnd = (x, y, t, zs)
    sc.params["t1"] = sc.t_end = T_END
    if sc.src is not None:
        sx, sy, _, q = sc.src
        sc.src = (sx, sy, np.array([0.0, T_END], np.float32), q * np.float32(min(1.0, n * m / 2.0 ** 22 + 0.02)))
    return sc


def _masked(case, seed):
    """A coast whose active area ends at ragged land and sea margins (so its uv-points are
    reached through index tables), with viscosity, Coriolis, wind, infiltration and the
    maximum velocity stored. The margin belongs to the mesh: it is the same for every seed."""
    sc = _regular(case, seed, viscosity=1, latitude=51.0, store_velmax=1)
    n, m = case["n"], case["m"]
    east = m - 2 - (0.2 * m * (0.5 + 0.5 * np.sin(np.arange(n) * (6.0 / n)))).astype(int)
    msk = sc.msk.reshape(m, n).copy()
    msk[np.arange(m)[:, None] > east[None, :]] = 0
    sc.msk = msk.reshape(-1)
    r = W.rng(seed + 1)
    tw = np.array([0.0, T_END], np.float32)
    sc.wind = (tw, np.full(2, r.uniform(8.0, 20.0), np.float32), np.full(2, 225.0, np.float32))
    if case.get("rain"):
        sc = W.with_infiltration(sc, qinf=3.0, qinf_zmin=0.0)
    return sc


def _quadtree(case, seed):
    """Four levels refined around the shoreline of a terrain that is the case's own; the
    surveyed bed, the tide and the wind are the seed's."""
    sc = W.quadtree_case(case["n"], case["m"], t_end=7200.0)
    r = W.rng(seed)
    sc.zb_qt = (sc.zb_qt + r.uniform(-0.2, 0.2, sc.zb_qt.shape)).astype(np.float32)
    t, zs = _tide(r.uniform(1.0, 3.0), r.uniform(0.0, 1.0))
    sc.bnd = (sc.bnd[0], sc.bnd[1], t, zs)
    sc.params["t1"] = sc.t_end = T_END
    sc.wind = (np.array([0.0, T_END], np.float32), np.full(2, r.uniform(10.0, 25.0), np.float32), sc.wind[2])
    return sc


def _member_cases(case, seed):
    """Sizes between the case's n and m, evenly in their logarithm, regular and subgrid in turn."""
    k = case["members"]
    out = []
    for j in range(k):
        f = j / max(k - 1, 1)
        size = int(round(math.exp(math.log(case["n"]) * (1 - f) + math.log(case["m"]) * f)))
        out.append(dict(mesh="subgrid" if j % 2 else "regular", n=size, m=size + j, rain=j % 4 == 0))
    return out


def _scenario(case, seed):
    if case["mesh"] == "regular":
        return _regular(case, seed, **({"use_qext": 1} if case.get("use") == "coupled" else {}))
    return {"subgrid": _subgrid, "masked": _masked, "quadtree": _quadtree}[case["mesh"]](case, seed)


def _qext(case, seed):
    """Exchange fluxes of a coupled model: up to 36 mm/h into a tenth of the cells."""
    r = W.rng(seed + 7)
    k = case["n"] * case["m"]
    return np.where(r.uniform(size=k) < 0.1, r.uniform(0.0, 1.0e-5, k), 0.0).astype(np.float32)


def _fields(case):
    out = ["zs", "zsmax"]
    if case.get("flow"):
        out += ["q", "uv"]
    if case["mesh"] == "masked":
        out += ["vmax"]
    return out


def prepare(case, seed):
    if case["use"] == "ensemble":
        batch = _lib.Batch()
        insts = []
        for j, c in enumerate(_member_cases(case, seed)):
            insts.append(_lib.Instance(_scenario(c, seed * 16 + j).build_model()))
            batch.add(insts[-1], T_END)
        return dict(case=case, batch=batch, insts=insts)
    state = dict(case=case, inst=_lib.Instance(_scenario(case, seed).build_model()))
    if case["use"] == "coupled":
        state["qext"] = _qext(case, seed)
    if case["use"] == "sweeps":
        state["t"], state["dt"] = 0.0, 1.0e-3
    return state


def run(state):
    case = state["case"]
    if case["use"] == "ensemble":
        batch = state["batch"]
        batch.advance(32)
        return [i.get("zs") for i in state["insts"] if not batch.done(i)]
    inst = state["inst"]
    if case["use"] == "coupled":
        inst.set("qext", state["qext"])
        inst.update(0.0)
        return dict(zs=inst.get("zs"))
    if case["use"] == "sweeps":
        dt = state["dt"]
        state["t"] += dt
        inst.update_forcing(state["t"], dt)
        min_dt = inst.compute_fluxes(dt)
        inst.compute_water_levels(state["t"], dt)
        state["dt"] = float(np.float32(0.5) * np.float32(min_dt))
        return dict(min_dt=min_dt, zs=inst.get("zs"))
    inst.update(case["span"])
    return {f: inst.get(f) for f in _fields(case)}


# ------------------------------------------------------------------------------------ work
def _mesh_work(mesh, cells, steps):
    """Bytes and operations of a pass of `steps` steps: the state and the tables of the wet part
    read once, the state written once (f64 levels and volumes, the rest f32), and about 120
    operations a uv-point and 20 a cell in each step. Two thirds of the coasts, a quarter of
    the fractal terrains and half of the quadtree cells are wet."""
    wet = {"regular": 0.66, "masked": 0.66, "subgrid": 0.25, "quadtree": 0.5}[mesh]
    cell = 16 + 8 + (16 + 8 + 12 + 8 if mesh == "subgrid" else 4)
    uv = 16 + 3 + (4 + 20 if mesh == "subgrid" else 8)
    if mesh in ("quadtree", "masked"):
        cell, uv = cell + 16, uv + 40
    return wet * cells * (cell + 2 * uv), wet * cells * steps * (20 + 2 * 120)


def _steps(case):
    if case["use"] in ("coupled", "sweeps"):
        return 1
    if case["use"] == "ensemble":
        return 32
    # the CFL step of the deepest water (10 m, 15 m of the fractal terrains)
    dx, h = {"regular": (50.0, 10.0), "masked": (50.0, 10.0), "subgrid": (25.0, 15.0), "quadtree": (12.5, 8.0)}[case["mesh"]]
    return max(1, round(case["span"] / (0.5 * dx / math.sqrt(9.81 * h))))


def work(case):
    if case["use"] == "ensemble":
        parts = [(c["mesh"], c["n"] * c["m"]) for c in _member_cases(case, 0)]
    else:   # a cell of the coarsest quadtree level holds about 40 cells
        parts = [(case["mesh"], case["n"] * case["m"] * (40 if case["mesh"] == "quadtree" else 1))]
    b, f = 0.0, 0.0
    for mesh, cells in parts:
        wb, wf = _mesh_work(mesh, cells, _steps(case))
        b, f = b + wb + 8.0 * cells, f + wf    # the levels are handed to the host once
    return dict(bytes=b, flops=f)


# ------------------------------------------------------- the same passes in 64-bit arithmetic
class _Points:
    """What the subgrid table recipe asks of a model: the order of a full rectangle's points
    (per cell the point on its right, then the one above)."""

    def __init__(self, n, m):
        c = np.arange(n * m)
        nn, mm = c % n, c // n
        has = np.stack([mm < m - 1, nn < n - 1], 1).reshape(-1)
        self.t = dict(uv_index_z_nm=(np.repeat(c, 2)[has] + 1).astype(np.int32),
                      uv_flags_dir=np.tile(np.array([0, 1], np.int8), n * m)[has],
                      z_index_z_n=(nn + 1).astype(np.int32), z_index_z_m=(mm + 1).astype(np.int32))

    def table(self, name):
        return self.t[name]


class _Exact:
    """The explicit step on a full rectangle in float64 torch: arrays [m, n], the points of the
    second direction as transposed views, so that axis 0 runs along a point's direction."""

    def __init__(self, sc, dev):
        self.dev, self.n, self.m = dev, sc.nmax, sc.mmax
        f32 = lambda v: float(np.float32(v))   # parameters as the scenario holds them
        p = sc.params
        self.g, self.dx = f32(9.81), f32(sc.dx)
        self.dxinv, self.area = f32(1.0 / np.float32(sc.dx)), f32(np.float32(sc.dx) * np.float32(sc.dx))
        self.kcs = self._cells(sc.msk).to(torch.int32)
        self.bt, self.bz = sc.bnd[2].astype(np.float64), sc.bnd[3][:, 0].astype(np.float64)
        self.rain = None if sc.rain is None else [np.asarray(a, np.float64) for a in sc.rain]
        self.qext = None
        self.sub = sc.subgrid is not None
        self.huth = 0.0 if self.sub else f32(0.05)
        if self.sub:
            self._tables(sc)
        else:
            self.zb = self._cells(sc.zb_grid)
            gn2 = f32(np.float32(9.81) * (np.float32(p["manning"]) * np.float32(p["manning"])))
            self.floor = [self._pair(a, torch.maximum) + self.huth for a in self._views(self.zb)]
            self.mean = [self._pair(a, lambda x, y: 0.5 * (x + y)) for a in self._views(self.zb)]
            self.gn2 = gn2
        bed = self.zmin if self.sub else self.zb
        self.zs = torch.clamp(bed, min=0.0)
        self.zsmax = torch.full_like(bed, -999.0)
        self.zs0, self.zsd = self.zs.clone(), torch.zeros_like(bed)
        if self.sub:
            self._volumes()
        self.src = None
        if sc.src is not None:
            c = (torch.from_numpy((np.floor(sc.src[0].astype(np.float64) / sc.dx) * self.n +
                                   np.floor(sc.src[1].astype(np.float64) / sc.dx)).astype(np.int64)).to(dev))
            q = torch.from_numpy(sc.src[3][0].astype(np.float64)).to(dev)
            self.src = torch.zeros(self.n * self.m, dtype=torch.float64, device=dev).index_add_(0, c, q).view(self.m, self.n)
        z = lambda a: torch.zeros_like(a)
        self.q = [z(bed), z(bed).t().contiguous()]
        self.u = [z(bed), z(bed).t().contiguous()]
        self.kf = [z(bed).bool(), z(bed).t().contiguous().bool()]
        # kinds of points: 1 computed, 2 boundary (between a boundary and an interior cell)
        self.k1, self.k2, self.dir = [], [], []
        for a in self._views(self.kcs):
            b = torch.cat([a[1:], torch.zeros_like(a[:1])])
            self.k1.append((a == 1) & (b == 1))
            self.k2.append(((a == 1) & (b == 2)) | ((a == 2) & (b == 1)))
            self.dir.append(torch.where(a == 2, 1.0, -1.0).to(torch.float64))
        self.adv = []
        for d in (0, 1):
            near = [self._sh(self.k1[d], -1, 0), self._sh(self.k1[d], 1, 0)]
            near += [self._self(self.k1[d], -1), self._self(self.k1[d], 1)]
            x = self.k1[1 - d].t()
            near += [x, self._sh(x, 0, -1), self._sh(x, 1, 0), self._sh(x, 1, -1)]
            ok = self.k1[d].clone()
            for v in near:
                ok &= v
            self.adv.append(ok)
        self.um = [z(v) for v in self.q]
        self.t, self.mindt = 0.0, 1.0e-6
        hc = f32(0.1)
        self.dtmax = min(60.0, 0.5 * self.dx / math.sqrt(9.81 * hc))

    def _cells(self, a):
        a = np.asarray(a)
        t = torch.from_numpy(np.ascontiguousarray(a.reshape(self.m, self.n))).to(self.dev)
        return t.double() if a.dtype.kind == "f" else t

    @staticmethod
    def _views(a):
        return a, a.t().contiguous()

    @staticmethod
    def _pair(a, op):
        return torch.cat([op(a[:-1], a[1:]), a[-1:]])

    @staticmethod
    def _sh(a, i, j):
        """a[k + i, l + j], zero (false) outside."""
        b = torch.zeros_like(a)
        s = lambda o, k: (slice(max(0, -o), k - max(0, o)), slice(max(0, o), k - max(0, -o)))
        (d0, s0), (d1, s1) = s(i, a.shape[0]), s(j, a.shape[1])
        b[d0, d1] = a[s0, s1]
        return b

    @staticmethod
    def _self(a, j):
        """a[k, l + j], the point itself outside."""
        return torch.cat([a[:, :1], a[:, :-1]], 1) if j < 0 else torch.cat([a[:, 1:], a[:, -1:]], 1)

    def _tables(self, sc):
        n, m, dev = self.n, self.m, self.dev
        pts = _Points(n, m)
        sg = sc.subgrid(pts)
        self.nl = nl = sg["nlevels"]
        self.zmin, self.zmax, self.volmax = (self._cells(sg[k]) for k in ("z_zmin", "z_zmax", "z_volmax"))
        self.zmax = torch.where(self.zmax - self.zmin <= 0, self.zmax + 0.01, self.zmax)
        self.dep = torch.from_numpy(np.ascontiguousarray(sg["z_level"])).to(dev).double().view(m, n, nl)
        nm = torch.from_numpy(pts.t["uv_index_z_nm"].astype(np.int64) - 1).to(dev)
        way = torch.from_numpy(pts.t["uv_flags_dir"]).to(dev)
        self.floor, self.umax, self.navg, self.fit, self.lev = [], [], [], [], []
        for d in (0, 1):
            sel = way == d
            c = nm[sel]

            def plane(name, width=1, sel=sel, c=c, d=d):
                v = torch.from_numpy(np.ascontiguousarray(sg[name])).to(dev).view(-1, width)[sel].double()
                out = torch.zeros(m * n, width, dtype=torch.float64, device=dev)
                out[c] = v
                out = out.view(m, n, width)
                out = out if d == 0 else out.transpose(0, 1).contiguous()
                return out[..., 0] if width == 1 else out
            zmin, zmax = plane("uv_zmin"), plane("uv_zmax")
            zmax = torch.maximum(zmax, zmin + 0.01)
            zmin = torch.maximum(zmin, self._pair(self._views(self.zmin)[d], torch.maximum))
            zmax = torch.maximum(zmax, zmin + 0.01)
            self.floor.append(zmin)
            self.umax.append(zmax)
            self.navg.append(self.g * plane("uv_navg").clamp(min=1e-4) ** 2)
            self.fit.append(plane("uv_ffit"))
            self.lev.append((plane("uv_havg", nl), self.g * plane("uv_nrep", nl).clamp(min=1e-4) ** 2, plane("uv_pwet", nl)))

    def _at(self, tab, k):
        return tab.gather(-1, k.unsqueeze(-1))[..., 0]

    def _volumes(self):
        above = self.zs >= self.zmax
        k = (self.dep > self.zs.unsqueeze(-1)).double()
        k[..., 0] = 0.0
        k = (torch.argmax(k, -1) - 1).clamp(min=0)
        d0, d1 = self._at(self.dep, k), self._at(self.dep, k + 1)
        dv = self.volmax / (self.nl - 1)
        part = (k + (self.zs - d0) / (d1 - d0).clamp(min=0.001)) * dv
        self.vol = torch.where(above, self.volmax + self.area * (self.zs - self.zmax.clamp(min=-20.0)), part)

    def _depth(self, d, z):
        """Flow depth, roughness term and wet fraction of direction d's points at level z."""
        lo, hi = self.floor[d], self.umax[d]
        havg, nrep, pwet = self.lev[d]
        full = z > hi
        top = havg[..., -1] - hi + z
        rough = self.navg[d] - (self.navg[d] - nrep[..., -1]) / (self.fit[d] * (z - hi).clamp(min=0.0) + 1.0)
        dz = (hi - lo) / (self.nl - 1)
        dz = torch.where(dz > 0, dz, torch.ones_like(dz))
        k = ((z - lo) / dz).floor().clamp(0, self.nl - 2).long()
        f = (z - (lo + k * dz)) / dz
        mix = lambda tab: self._at(tab, k) + (self._at(tab, k + 1) - self._at(tab, k)) * f
        one = torch.ones_like(z)
        return (torch.where(full, top, mix(havg)), torch.where(full, rough, mix(nrep)), torch.where(full, one, mix(pwet)))

    def forcing(self, t, dt):
        """Weakly reflective water-level boundary at time t (step dt)."""
        level = float(np.interp(t, self.bt, self.bz))
        bed = self.zmin if self.sub else self.zb
        zsb = torch.clamp(bed, min=level)
        factime = min(dt / 60.0, 1.0)
        facrel = 1.0 - min(dt / 3600.0, 1.0)
        vol = self.vol if self.sub else None
        for d in (0, 1):
            sel = self.k2[d]
            if not bool(sel.any()):
                continue
            t_ = (lambda a: a) if d == 0 else (lambda a: a.t())
            zs, zb_, bd = t_(self.zs), t_(zsb), t_(bed)
            west = self.dir[d] > 0                       # the boundary cell is the first one
            up = lambda a: torch.cat([a[1:], a[-1:]])
            pick = lambda a: torch.where(west, up(a), a)  # the interior cell's value
            here = lambda a: torch.where(west, a, up(a))  # the boundary cell's value
            zi, zo, bo = pick(zs), here(zb_), here(bd)
            if self.sub:
                z = torch.maximum(zo, zi)
                h = self._depth(d, z)[0]
                h = torch.where(z > self.floor[d], h, torch.zeros_like(h)).clamp(min=self.huth)
                dry_in = pick(t_(vol)) <= 0.0
            else:
                h = (0.5 * (zo + zi) - self.mean[d]).clamp(min=self.huth)
                dry_in = zi - pick(bd) <= self.huth
            dry = h < self.huth + 1e-6
            hs = torch.where(dry, torch.ones_like(h), h)
            qb = -self.dir[d] * torch.sqrt(self.g / hs) * (zi - zo) * hs + self.um[d]
            out = lambda v: torch.where(west, v.clamp(max=0.0), v.clamp(min=0.0))
            inn = lambda v: torch.where(west, v.clamp(min=0.0), v.clamp(max=0.0))
            qb = torch.where(dry_in, inn(qb), qb)
            qb = torch.where(zo - bo < self.huth, out(qb), qb)
            qb = torch.where(dry, torch.zeros_like(qb), qb)
            um = torch.where(dry, torch.zeros_like(qb), self.um[d])
            self.q[d] = torch.where(sel, qb, self.q[d])
            self.u[d] = torch.where(sel, (qb / hs).clamp(-4.0, 4.0), self.u[d])
            self.um[d] = torch.where(sel, factime * qb + facrel * (1.0 - factime) * um, self.um[d])
        b = self.kcs == 2
        self.zs = torch.where(b, zsb, self.zs)
        self.zsmax = torch.where(b, torch.maximum(self.zsmax, self.zs), self.zsmax)

    def momentum(self, dt):
        most, new = 0.0, []
        for d in (0, 1):
            t_ = (lambda a: a) if d == 0 else (lambda a: a.t())
            zs = t_(self.zs)
            zu = torch.cat([zs[1:], zs[-1:]])
            z = torch.maximum(zs, zu)
            wet = self.k1[d] & (z > self.floor[d])
            if self.sub:
                hu, gn2, phi = self._depth(d, z)
            else:
                hu, gn2, phi = (z - self.floor[d]).clamp(min=self.huth), torch.full_like(z, self.gn2), torch.ones_like(z)
            hu = torch.where(wet, hu, torch.ones_like(hu))
            q, u, sh = self.q[d], self.u[d], self._sh
            qx, ux = self.q[1 - d].t(), self.u[1 - d].t()
            slope = (zu - zs) * self.dxinv
            frc = -self.g * hu * slope
            eps, di = 1.0e-6, self.dxinv
            qd, qu = (sh(q, -1, 0) + q) / 2, (q + sh(q, 1, 0)) / 2
            ud, uu = (sh(u, -1, 0) + u) / 2, (u + sh(u, 1, 0)) / 2
            zero = torch.zeros_like(q)
            a = torch.where(qd > eps, (qd * (u - sh(u, -1, 0)) + ud * (q - sh(q, -1, 0))) * di, zero)
            a = a + torch.where(qu < -eps, (qu * (sh(u, 1, 0) - u) + uu * (sh(q, 1, 0) - q)) * di, zero)
            yn, yd = (qx + sh(qx, 1, 0)) / 2, (sh(qx, 0, -1) + sh(qx, 1, -1)) / 2
            a = a + torch.where(yd > eps, yd * (u - self._self(u, -1)) * di, zero)
            a = a + torch.where(yn < -eps, yn * (self._self(u, 1) - u) * di, zero)
            a = a + torch.where(ud > eps, ud * (qx - sh(qx, 0, -1)) * di, zero)
            a = a + torch.where(uu < -eps, uu * (sh(qx, 1, 0) - sh(qx, 1, -1)) * di, zero)
            adv = torch.minimum(torch.maximum(-phi * a, -hu), hu)
            frc = frc + torch.where(self.adv[d], adv, zero)
            vu = (sh(ux, 0, -1) + sh(ux, 1, -1) + ux + sh(ux, 1, 0)) / 4
            start = torch.sqrt(slope.abs() / (gn2.clamp(min=1e-5) / 10.0)) * hu ** (5.0 / 3.0)
            qfr = torch.where(self.kf[d], torch.sqrt(q * q + (hu * vu) ** 2), start)
            qn = (q + frc * dt) / (1.0 + gn2 * dt * qfr / hu ** (7.0 / 3.0))
            if self.sub:
                zd, v = t_(self.zsd), t_(self.vol)
                rough = (zd - torch.cat([zd[1:], zd[-1:]])).abs() - 0.1
                qn = torch.where(rough > 0, qn * 0.1 / (0.1 * rough + 0.1), qn)
                low, high = v < 0, torch.cat([v[1:], v[-1:]]) < 0
            else:
                zb = t_(self.zb)
                low, high = zs < zb, zu < torch.cat([zb[1:], zb[-1:]])
            qn = torch.where(low, qn.clamp(max=0.0), qn)
            qn = torch.where(high, qn.clamp(min=0.0), qn)
            qn = torch.minimum(torch.maximum(qn, -10.0 * hu), 10.0 * hu)
            un = qn / hu
            den = torch.where(wet, torch.maximum(torch.sqrt(self.g * hu), un.abs()) * di, zero)
            most = max(most, float(den.max()))
            keep = ~self.k1[d]
            new.append((torch.where(keep, q, torch.where(wet, qn, zero)), torch.where(keep, u, torch.where(wet, un, zero)), wet))
        for d in (0, 1):
            self.q[d], self.u[d], self.kf[d] = new[d]
        self.mindt = min(self.dtmax, 1.0 / most) if most > 0 else self.dtmax

    def continuity(self, t, dt):
        u, v = self.q[0], self.q[1].t()
        net = (self._sh(u, -1, 0) - u) + (self._sh(v, 0, -1) - v)
        gain = 0.0
        if self.rain is not None:
            gain = float(np.interp(t, *self.rain)) / 3.6e6
        if self.qext is not None:
            gain = gain + self.qext
        one = self.kcs == 1
        if self.sub:
            vol = self.vol if self.src is None else self.vol + torch.where(self.vol >= 0, self.src * dt, torch.zeros_like(self.vol))
            vol = torch.where(one, vol + (net * self.dx + gain * self.area) * dt, vol)
            dv = self.volmax / (self.nl - 1)
            k = (vol / dv).floor().clamp(0, self.nl - 2).long()
            d0, d1 = self._at(self.dep, k), self._at(self.dep, k + 1)
            z = d0 + (d1 - d0) * (vol - k * dv) / dv
            z = torch.where(vol <= 1e-6, self.zmin.clamp(min=-20.0), z)
            z = torch.where(vol >= 0.999 * self.volmax, self.zmax.clamp(min=-20.0) + (vol - self.volmax) / self.area, z)
            self.vol = vol
            z = torch.where(one, z, self.zs)
            self.zsd = torch.where(one, z - 2.0 * self.zs + self.zs0, self.zsd)
            self.zs0 = torch.where(one, self.zs, self.zs0)
            self.zs = z
        else:
            self.zs = torch.where(one, self.zs + (gain + net * self.dxinv) * dt, self.zs)
        self.zsmax = torch.maximum(self.zsmax, self.zs)

    def step(self):
        dt = 0.5 * self.mindt
        self.t += dt
        self.forcing(self.t, dt)
        self.momentum(dt)
        self.continuity(self.t, dt)

    def points(self, planes):
        """Discharges or velocities in the order a program reads them, the dummy last."""
        m, n = self.m, self.n
        both = torch.stack([planes[0], planes[1].t()], -1)
        has = torch.ones(m, n, 2, dtype=torch.bool, device=self.dev)
        has[-1, :, 0] = False
        has[:, -1, 1] = False
        return torch.cat([both[has], torch.zeros(1, dtype=torch.float64, device=self.dev)])


def _exact_pass(case, seed, steps=None):
    sc = _scenario(case, seed)
    e = _Exact(sc, torch.device("cuda" if torch.cuda.is_available() else "cpu"))
    if case.get("use") == "coupled":
        e.qext = e._cells(_qext(case, seed))
        steps = 1
    if steps is not None:
        for _ in range(steps):
            e.step()
    else:
        while e.t < case["span"]:
            e.step()
    return e


def exact(case, seed):
    if case["mesh"] in ("quadtree", "masked"):
        return None      # index tables of the mesh are the framework's own work
    if case["use"] == "ensemble":
        return [_exact_pass(c, seed * 16 + j, 32).zs.reshape(-1) for j, c in enumerate(_member_cases(case, seed))]
    if case["use"] == "sweeps":
        sc = _scenario(case, seed)
        e = _Exact(sc, torch.device("cuda" if torch.cuda.is_available() else "cpu"))
        dt = float(np.float32(1.0e-3))
        e.forcing(1.0e-3, dt)
        e.momentum(dt)
        e.continuity(1.0e-3, dt)
        return dict(min_dt=e.mindt, zs=e.zs.reshape(-1))
    e = _exact_pass(case, seed)
    if case["use"] == "coupled":
        return dict(zs=e.zs.reshape(-1))
    out = dict(zs=e.zs.reshape(-1), zsmax=e.zsmax.reshape(-1))
    if case.get("flow"):
        out.update(q=e.points(e.q), uv=e.points(e.u))
    return out
