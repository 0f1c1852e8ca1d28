"""The work a user of this framework has it do, as cases that can be timed.

Every case is one whole forecast through the public Python entry points: the
layers are registered from host arrays (bathymetry and initial elevation),
the root steps run on the device, and the state and the maximum/arrival
fields come back to the host.  `prepare` makes the host arrays a user's
program holds before the call, `run` is the call.

Kinds of case:
  single   DeviceRun of one layer: linear or nonlinear, spherical or
           Cartesian, the whole-run device loop
  nest     DeviceRun of a spherical linear parent with a Cartesian nonlinear
           child (REL_SIZE / REL_TIME)
  source   an Okada fault on a layer, then the loop with tide gauges sampled
           after every step
  dropin   the reference's per-call entry sequence, call by call
  batch    many scenarios of uneven sizes through the batch engine, in chunks
           as the serving loop runs them
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gpu-comcot_amd"))

from gcomcot import DeviceRun, LayerSpec, Scenario  # noqa: E402
from gcomcot.batch import Batch  # noqa: E402
from gcomcot.source import Fault  # noqa: E402

F32 = np.float32
GRAV = float(F32(9.807))
R_EARTH = 6378000.0
RAD_MIN = float(F32(0.000290888208665721))
RAD_DEG = float(F32(0.01745329252))


def listed():
    return [
        # a coarse regional grid run for a quick look: launches and calls count
        dict(name="linear-96x72", kind="single", cord=0, gov=0, nx=96, ny=72, dx=4.0, steps=60),
        # the 2000-step single-layer linear configuration at 2 arc-minutes
        dict(name="linear-1024x768", kind="single", cord=0, gov=0, nx=1024, ny=768, dx=2.0, steps=2000),
        # a linear ocean basin whose sides are no multiple of anything
        dict(name="linear-2051x1537", kind="single", cord=0, gov=0, nx=2051, ny=1537, dx=1.0, steps=1000),
        # the largest linear grid: more than the last-level cache holds
        dict(name="linear-4096x3072", kind="single", cord=0, gov=0, nx=4096, ny=3072, dx=0.5, steps=1500),
        # a bay with a moving shoreline, odd sides, Manning friction
        dict(name="nonlinear-517x391", kind="single", cord=0, gov=1, nx=517, ny=391, dx=0.5, steps=400),
        # the headline configuration: nonlinear 4096x3072 with run-up and maxima
        dict(name="nonlinear-4096x3072", kind="single", cord=0, gov=1, nx=4096, ny=3072, dx=0.5, steps=1500),
        # a harbour model on a metre grid
        dict(name="nonlinear-cart-1201x901", kind="single", cord=1, gov=1, nx=1201, ny=901, dx=0.05, steps=800),
        # a small regional nest
        dict(name="nest-512x384+401", kind="nest", nx=512, ny=384, dx=2.0, foot=100, rs=4, rt=4, steps=300),
        # the two-level nest configuration: 2048x1536 parent, 1801x1801 child
        dict(name="nest-2048x1536+1801", kind="nest", nx=2048, ny=1536, dx=2.0, foot=450, rs=4, rt=4, steps=400),
        # an earthquake source computed on the device, forecast with 24 gauges
        dict(name="source-1024x768", kind="source", cord=0, gov=1, nx=1024, ny=768, dx=1.0, gauges=24, steps=300),
        # the Fortran driver's call sequence on a small nest: per-call latency
        dict(name="dropin-256x192+121", kind="dropin", nx=256, ny=192, dx=2.0, foot=40, rs=3, rt=3, steps=60),
        # a warning centre's batch: uneven scenarios, a quarter of them nested
        dict(name="batch-16", kind="batch", count=16, cells_lo=256 * 192, cells_hi=1365 * 1024, lo=200, hi=600),
    ]


def draw(rng):
    def logu(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    def sides(lo, hi):  # both sides from the cell count, odd as they come
        cells, asp = logu(lo, hi), rng.uniform(0.6, 1.7)
        return max(24, int(math.sqrt(cells * asp))), max(24, int(math.sqrt(cells / asp)))

    kind = rng.choice(["single", "single", "single", "nest", "source", "dropin", "batch"])
    if kind == "single":
        cord, gov = rng.choice([(0, 0), (0, 0), (0, 1), (0, 1), (1, 1)])
        nx, ny = sides(64 * 48, 3600 * 2700)
        dx = rng.choice([0.5, 1.0, 2.0]) if cord == 0 else 0.05
        return dict(kind=kind, cord=cord, gov=gov, nx=nx, ny=ny, dx=dx, steps=logu(40, 1000))
    if kind == "source":
        nx, ny = sides(128 * 96, 2048 * 1536)
        return dict(kind=kind, cord=0, gov=rng.choice([0, 1]), nx=nx, ny=ny, dx=1.0,
                    gauges=rng.randint(1, 40), steps=logu(50, 500))
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(3, 20), cells_lo=128 * 96, cells_hi=1024 * 768,
                    lo=rng.randint(50, 150), hi=rng.randint(200, 500))
    nx, ny = sides(*((256 * 192, 1600 * 1200) if kind == "nest" else (160 * 120, 512 * 384)))
    rs, rt = rng.randint(2, 5), rng.randint(2, 6)
    foot = max(8, int(min(nx, ny) * rng.uniform(0.15, 0.45)))
    return dict(kind=kind, nx=nx, ny=ny, dx=2.0, foot=min(foot, 1600 // rs), rs=rs, rt=rt,
                steps=logu(40, 300) if kind == "nest" else logu(10, 60))


# ------------------------------------------------------------------ inputs
class World:
    """A coast on the west side (bays, a shelf, an abyssal plain with
    seamounts) over the unit square, and one dipole or hump source."""

    def __init__(self, rng, width_km, height_km, nonlinear):
        self.w, self.h = width_km, height_km
        self.coast = rng.uniform(0.06, 0.14)
        self.bays = [(rng.uniform(0.01, 0.04), rng.uniform(1.0, 6.0), rng.uniform(0, 2 * math.pi)) for _ in range(3)]
        self.shelf = rng.uniform(0.10, 0.2)
        self.deep = rng.uniform(3000.0, 4800.0) if width_km > 300 else rng.uniform(40.0, 80.0)
        self.edge = min(180.0, self.deep * 0.3)
        self.mounts = [(rng.uniform(0.35, 0.95), rng.uniform(0.05, 0.95), rng.uniform(0.03, 0.08),
                        self.deep * rng.uniform(0.2, 0.6)) for _ in range(6)]
        self.peak = rng.uniform(0.8, 3.0) if width_km > 300 else rng.uniform(0.8, 2.0)
        self.sx, self.sy = rng.uniform(0.25, 0.6), rng.uniform(0.3, 0.7)
        self.sig = rng.uniform(0.04, 0.08)
        self.dipole = nonlinear

    def depth(self, u, v):
        """Still-water depth at the points v (rows) x u (columns) of the square, negative on land."""
        shore = self.coast + sum(a * np.sin(2 * math.pi * k * v + p) for a, k, p in self.bays)
        d = (u[None, :] - shore[:, None]).astype(F32)  # distance from the shore
        h = np.where(d < self.shelf, d * F32(self.edge / self.shelf),
                     F32(self.edge) + (d - F32(self.shelf)) * F32(6.0 * (self.deep - self.edge)))
        np.minimum(h, F32(self.deep), out=h)
        np.maximum(h, F32(-120.0), out=h)
        for x, y, s, top in self.mounts:
            gx = np.exp(-((u - x) / s) ** 2).astype(F32)
            gy = (top * np.exp(-((v - y) / (s * self.w / self.h)) ** 2)).astype(F32)
            deepm = h > F32(500.0) if self.deep > 500 else h > F32(30.0)
            h -= (gy[:, None] * gx[None, :]) * deepm
        return np.ascontiguousarray(h, F32)

    def eta(self, u, v, h):
        sv = self.sig * self.w / self.h
        gx = np.exp(-((u - self.sx) / self.sig) ** 2)
        if self.dipole:
            gx = gx - 0.8 * np.exp(-((u - self.sx - 2.2 * self.sig) / self.sig) ** 2)
        gy = self.peak * np.exp(-((v - self.sy) / sv) ** 2)
        z = gy.astype(F32)[:, None] * gx.astype(F32)[None, :]
        z[h <= 0] = 0.0
        return np.ascontiguousarray(z, F32)


def _root(rng, cord, gov, nx, ny, dx, zero=False):
    """An outermost layer and the world it lies in (dx in arc-minutes)."""
    lat0 = 5.0 if (ny - 1) * dx / 60.0 > 40.0 else float(rng.uniform(-15.0, 20.0))
    km = dx * 1.855
    w = World(rng, nx * km, ny * km, gov == 1)
    u, v = (np.arange(nx) + 0.5) / nx, (np.arange(ny) + 0.5) / ny
    h = w.depth(u, v)
    z = np.zeros_like(h) if zero else w.eta(u, v, h)
    lat = lat0 + np.arange(ny, dtype=np.float64) * dx / 60.0
    cos = math.cos(math.radians(max(abs(lat[0]), abs(lat[-1]))))
    dxm, dym = float(F32(R_EARTH * cos * dx * RAD_MIN)), float(F32(R_EARTH * dx * RAD_MIN))
    cfl = 0.35 if gov else 0.5
    dt = float(F32(cfl * min(dxm, dym) / math.sqrt(GRAV * float(h.max()))))
    fric = dict(fric_switch=0, fric_coef=0.013) if gov else dict(fric_switch=1, fric_coef=0.0)
    geo = dict(dx=float(F32(dx)), dy=float(F32(dx)), y=lat.astype(F32), dely=np.full(ny, dx, F32)) \
        if cord == 0 else dict(dx=dxm, dy=dym)
    return w, LayerSpec(id=1, parent=-1, level=1, laycord=cord, laygov=gov, nx=nx, ny=ny, dt=dt,
                        h=h, z0=z, **geo, **fric)


def _nest(rng, nx, ny, dx, foot, rs, rt, steps, name):
    """A linear spherical root and a nonlinear Cartesian child over its coast."""
    w, P = _root(rng, 0, 0, nx, ny, dx)
    foot_i = min(foot, nx - 12)
    foot_j = min(foot, ny - 12)
    i0, j0 = max(4, int(0.03 * nx)), max(4, (ny - foot_j) // 2)
    i1, j1 = min(i0 + foot_i - 1, nx - 4), j0 + foot_j - 1
    cnx, cny = (i1 - i0 + 1) * rs + 1, (j1 - j0 + 1) * rs + 1
    u = (i0 - 1 + (np.arange(cnx) - 0.5) / rs) / nx
    v = (j0 - 1 + (np.arange(cny) - 0.5) / rs) / ny
    h = w.depth(u, v)
    mid = math.radians(float(P.y[(j0 + j1) // 2 - 1]))
    C = LayerSpec(id=2, parent=1, level=2, laycord=1, laygov=1, nx=cnx, ny=cny,
                  dx=float(F32(R_EARTH * math.cos(mid) * dx * RAD_MIN / rs)),
                  dy=float(F32(R_EARTH * dx * RAD_MIN / rs)), dt=float(F32(F32(P.dt) / F32(rt))),
                  h=h, z0=w.eta(u, v, h), fric_switch=0, fric_coef=0.013, rel_size=rs, rel_time=rt,
                  corners=(i0, i1, j0, j1))
    return Scenario(name, [P, C], steps)


def _scenarios(case, seed):
    rng = np.random.default_rng(seed)
    k = case["kind"]
    if k in ("single", "source"):
        _, L = _root(rng, case["cord"], case["gov"], case["nx"], case["ny"], case["dx"], zero=k == "source")
        return [Scenario(k, [L], case["steps"])]
    if k in ("nest", "dropin"):
        return [_nest(rng, case["nx"], case["ny"], case["dx"], case["foot"], case["rs"], case["rt"],
                      case["steps"], k)]
    # batch: sizes and step counts belong to the case (they are its work);
    # bathymetry and sources to the seed
    shapes = np.random.default_rng(case["count"] * 1000 + case["hi"])
    out = []
    for q in range(case["count"]):
        ny = int(math.sqrt(0.75 * math.exp(shapes.uniform(math.log(case["cells_lo"]), math.log(case["cells_hi"])))))
        nx, dx = ny * 4 // 3, float(shapes.choice([1.0, 2.0]))
        steps, rs = int(shapes.integers(case["lo"], case["hi"] + 1)), int(shapes.choice([3, 4, 5]))
        side = int(shapes.uniform(200, 700))
        if q % 4 == 0:
            out.append(_nest(rng, nx, ny, dx, max(8, min(side // rs, nx // 2, ny // 2)), rs, rs, steps, f"b{q}"))
        else:
            out.append(Scenario(f"b{q}", [_root(rng, 0, 0, nx, ny, dx)[1]], steps))
    return out


def prepare(case, seed):
    state = dict(case=case, scenarios=_scenarios(case, seed))
    if case["kind"] == "source":
        L, rng = state["scenarios"][0].layers[0], np.random.default_rng(seed + 1)
        x = np.arange(L.nx) * L.dx / 60.0
        size = float(rng.uniform(0.6, 1.0)) * min(300e3, 0.25 * L.nx * L.dx * 1855.0)
        state["fault"] = Fault(float(rng.uniform(5e3, 15e3)), size, 0.4 * size, float(rng.uniform(3, 8)),
                               float(rng.uniform(0, 60)), float(rng.uniform(10, 30)), 90.0,
                               x0=float(F32(x[int(0.45 * L.nx)])), y0=float(L.y[L.ny // 2]))
        state["gauges"] = [(float(F32(x[1] + rng.uniform(0.02, 0.95) * (x[-1] - x[1]))),
                            float(F32(L.y[0] + rng.uniform(0.03, 0.97) * (L.y[-1] - L.y[0]))), 1)
                           for _ in range(case["gauges"])]
    return state


# --------------------------------------------------------------------- run
def _fields(run, sc):
    out = {}
    for L in sc.layers:
        s, m = run.state(L.id), run.maxima(L.id)
        out[f"layer{L.id}"] = {"z": s["z1"], "m": s["m1"], "n": s["n1"],
                               "zmax": m["zmax_wet"], "arrival": m["arrival"]}
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        b = Batch()
        sids = [b.add(sc) for sc in state["scenarios"]]
        out = {}
        while sids:
            b.run(128)
            for sid in b.finished():
                m = b.maxima(sid, 1)
                out[f"s{b.specs[sid].name}"] = {"zmax": m["zmax_wet"], "arrival": m["arrival"]}
                b.remove(sid)
                sids.remove(sid)
        b.close()
        return out
    sc = state["scenarios"][0]
    r = DeviceRun(sc)
    out = {}
    if case["kind"] == "source":
        r.set_coords()
        r.fault(state["fault"].params(), state["fault"].switch)
        r.set_gauges(state["gauges"], case["steps"])
        r.run(case["steps"])
        out["gauges"] = r.gauges(case["steps"])
    elif case["kind"] == "dropin":
        for _ in range(case["steps"]):
            r.dropin_step()
    else:
        r.run(case["steps"])
    out.update(_fields(r, sc))
    r.close()
    return out


def work(case):
    """Inputs (depth, elevation) read once, outputs (five planes a layer, two
    a batched scenario) written once; the arithmetic of every cell update: 26
    operations linear, 150 nonlinear."""
    total, flops = 0.0, 0.0
    if case["kind"] == "batch":
        for sc in _sizes(case):
            total += sum(8.0 * c for c, _, _ in sc[0]) + 8.0 * sc[0][0][0]
            flops += sc[1] * sum(c * sub * f for c, sub, f in sc[0])
        return {"bytes": total, "flops": flops}
    if case["kind"] in ("single", "source"):
        layers = [(case["nx"] * case["ny"], 1, 150 if case["gov"] else 26)]
    else:
        side = case["foot"] * case["rs"] + 1
        layers = [(case["nx"] * case["ny"], 1, 26), (side * side, case["rt"], 150)]
    return {"bytes": sum(28.0 * c for c, _, _ in layers),
            "flops": float(case["steps"] * sum(c * s * f for c, s, f in layers))}


def _sizes(case):
    """Cells, sub-steps and operations of a batch's layers, and its step counts."""
    shapes = np.random.default_rng(case["count"] * 1000 + case["hi"])
    out = []
    for q in range(case["count"]):
        ny = int(math.sqrt(0.75 * math.exp(shapes.uniform(math.log(case["cells_lo"]), math.log(case["cells_hi"])))))
        nx = ny * 4 // 3
        shapes.choice([1.0, 2.0])
        steps, rs = int(shapes.integers(case["lo"], case["hi"] + 1)), int(shapes.choice([3, 4, 5]))
        side = int(shapes.uniform(200, 700))
        layers = [(nx * ny, 1, 26)]
        if q % 4 == 0:
            layers.append(((max(8, min(side // rs, nx // 2, ny // 2)) * rs + 1) ** 2, rs, 150))
        out.append((layers, steps))
    return out


# ------------------------------------------------------------------- exact
# The same equations in 64 bits on whole planes with plain torch: COMCOT's
# staggered leapfrog (continuity, radiating boundary, momentum, nesting).
GX, EPS, LAND, VLIM, SPAN = float(F32(1e-5)), float(F32(1e-10)), -50.0, 20.0, 10
MAN = float(F32(2.3333333))


def _sh(a, dj, di):
    """a at (j + dj, i + di), the nearest cell beyond the edges."""
    if di:
        a = torch.cat([a[:, 1:], a[:, -1:]], 1) if di > 0 else torch.cat([a[:, :1], a[:, :-1]], 1)
    if dj:
        a = torch.cat([a[1:], a[-1:]], 0) if dj > 0 else torch.cat([a[:1], a[:-1]], 0)
    return a


class _Exact:
    def __init__(self, s, dev):
        t = lambda a: torch.from_numpy(np.array(a, np.float64)).to(dev)  # noqa: E731
        self.s, self.h, self.z = s, t(s.h), t(s.z0)
        self.root, self.nl, self.sph = s.id == 1, s.laygov == 1, s.laycord == 0
        z = torch.zeros_like
        self.m, self.n, self.zmax = z(self.h), z(self.h), z(self.h)
        self.dz = z(self.h)
        dt = s.dt
        if self.sph:
            y, d = t(s.y)[:, None], t(s.dely)[:, None]
            am, an = y * RAD_DEG, (y + 0.5 * d * float(F32(0.016666666667))) * RAD_DEG
            rr = dt / R_EARTH
            rt = 0.5 * dt * float(F32(7.2722e-5))
            ex, ey = s.dx * RAD_MIN, d * RAD_MIN
            self.r1, self.r11, self.r6 = rr / torch.cos(am) / ex, rr / torch.cos(am) / ey, torch.cos(an)
            self.px, self.py = GRAV * self.r1, GRAV * rr / ey
            self.ax, self.axc = self.r1, rr / ey           # advection: x equation along, across
            self.ay, self.ayc = rr / ey, rr / torch.cos(an) / ex
            self.cx, self.cy = rt * torch.sin(am), -rt * torch.sin(an)
        else:
            rx, ry = dt / s.dx, dt / s.dy
            self.r1, self.r11, self.r6 = rx, ry, 1.0
            self.px, self.py, self.ax, self.axc, self.ay, self.ayc = GRAV * rx, GRAV * ry, rx, ry, ry, rx
            self.cx = self.cy = 0.0
        self.kf = 0.5 * dt * GRAV * s.fric_coef ** 2 if s.fric_switch == 0 else 0.0
        ny, nx = self.h.shape
        self.out = torch.ones_like(self.h, dtype=torch.bool)   # momentum's range, both directions
        self.out[:, -1] = False
        self.out[-1] = False
        self.okx, self.oky = self.out.clone(), self.out.clone()
        if not self.nl:
            self.okx[-1], self.oky[:, -1] = True, True
            self.okx[:, -1], self.oky[-1] = False, False
        if not self.root:
            for a in (self.okx, self.oky):
                a[0], a[:, 0] = False, False
            self.okx[-1, 1:-1], self.oky[1:-1, -1] = True, True
        self.core = torch.zeros_like(self.out)
        self.core[SPAN:ny - SPAN - 1, SPAN:nx - SPAN - 1] = True

    def mass(self):
        h, z, m, n = self.h, self.z, self.m, self.n
        r6 = self.r6 if self.sph else torch.ones_like(h[:, :1])
        zz = z - self.r1 * (m - _sh(m, 0, -1)) - self.r11 * (n * r6 - _sh(n * r6, -1, 0))
        zz = torch.where(zz.abs() < EPS, 0.0, zz)
        if self.nl:
            dd = zz + h
            wet = ((h >= LAND) if self.sph else (h > LAND)) & (dd >= GX)
            self.dz, z2 = torch.where(wet, dd, 0.0), torch.where(wet, zz, -h)
        else:
            z2 = torch.where(h > GX, torch.where(zz + h <= EPS, -h, zz), 0.0)
        if self.root:
            for sl, z_ring in self.ring():
                z2[sl] = z_ring
                self.dz[sl] = 0.0
        else:
            self.dz[0], self.dz[:, 0] = 0.0, 0.0
            z2[0], z2[:, 0] = 0.0, 0.0
        self.z2 = z2

    def ring(self):
        h, m, n = self.h, self.m, self.n

        def rad(hh, q, neg):
            zz = torch.sqrt(q) / torch.sqrt(GRAV * hh.clamp_min(GX))
            zz = torch.where(neg, -zz, zz)
            return torch.where((hh > GX) & (zz.abs() <= 99.0), zz, 0.0)

        a = slice(1, -1)
        uh = 0.5 * (m[0, 1:-1] + m[0, :-2])
        yield (0, a), rad(h[0, a], uh ** 2 + n[0, a] ** 2, n[0, a] > 0)
        uh = 0.5 * (m[-1, 1:-1] + m[-1, :-2])
        yield (-1, a), rad(h[-1, a], uh ** 2 + n[-2, a] ** 2, n[-2, a] < 0)
        uh = torch.where(h[:-2, 0] > GX, 0.5 * (n[1:-1, 0] + n[:-2, 0]), n[1:-1, 0])
        yield (a, 0), rad(h[a, 0], uh ** 2 + m[a, 0] ** 2, m[a, 0] > 0)
        uh = 0.5 * (n[1:-1, -1] + n[:-2, -1])
        yield (a, -1), rad(h[a, -1], uh ** 2 + m[a, -2] ** 2, m[a, -2] < 0)
        for j, i, q, p, neg in ((0, 0, m[0, 0], n[0, 0], (m[0, 0] > 0) | (n[0, 0] > 0)),
                                (0, -1, m[0, -2], n[0, -1], (m[0, -2] < 0) | (n[0, -1] > 0)),
                                (-1, 0, m[-1, 0], n[-2, 0], (m[-1, 0] > 0) | (n[-2, 0] < 0)),
                                (-1, -1, m[-1, -2], n[-2, -1], (m[-1, -2] < 0) | (n[-2, -1] < 0))):
            yield (j, i), rad(h[j, i], q ** 2 + p ** 2, neg)

    def momentum(self):
        z2, h = self.z2, self.h
        if self.nl:
            dzdt = (z2 - self.z).abs() / self.s.dt
            c = torch.sqrt(GRAV * self.dz)
            brk = torch.where(dzdt > 0.08 * c, torch.exp(-(dzdt - 0.08 * c) / ((0.65 - 0.08) * c)), 1.0)
            T = lambda a: a.t().contiguous() if torch.is_tensor(a) else a  # noqa: E731
            x = self.flux(self.m, self.n, z2, h, self.dz, brk, self.px, self.ax, self.axc, self.cx, True, self.core)
            y = T(self.flux(T(self.n), T(self.m), T(z2), T(h), T(self.dz), T(brk), T(self.py), T(self.ay),
                            T(self.ayc), T(self.cy), self.sph, T(self.core)))
        else:
            hp, hq = _sh(h, 0, 1), _sh(h, 1, 0)
            m, n = self.m, self.n
            tn = n + _sh(n, 0, 1) + _sh(n, -1, 0) + _sh(n, -1, 1)
            x = m - self.px * 0.5 * (h + hp) * (_sh(z2, 0, 1) - z2) + self.cx * tn
            x = torch.where((h > GX) & (hp > GX) & (x.abs() >= EPS), x, 0.0)
            tm = m + _sh(m, 1, 0) + _sh(m, 0, -1) + _sh(m, 1, -1)
            y = n - self.py * 0.5 * (h + hq) * (_sh(z2, 1, 0) - z2) + self.cy * tm
            y = torch.where((h > GX) & (hq > GX) & (y.abs() >= EPS), y, 0.0)
        self.m2, self.n2 = torch.where(self.okx, x, 0.0), torch.where(self.oky, y, 0.0)
        wet = h + z2 > GX
        if not self.root:
            wet[0], wet[:, 0] = False, False
        self.zmax = torch.where(wet & (z2 > self.zmax), z2, self.zmax)

    def flux(self, p, q, z, h, dz, brk, press, fa, fc, cor, fric, core):
        """Nonlinear flux along the second axis (p) with the cross flux q."""
        he, ze, dze = _sh(h, 0, 1), _sh(z, 0, 1), _sh(dz, 0, 1)
        hp = torch.where(h > GX, 0.5 * (h + he), 0.0)
        cut = lambda v: torch.where(v < GX, 0.0, v)  # noqa: E731
        d1, d2 = cut(0.25 * (dz + dze)), cut(0.5 * (dz + dze))
        both = (dz > GX) & (dze > GX)
        out = (dz > GX) & (dze <= GX) & (he + z > GX)
        inn = (dz <= GX) & (dze > GX) & (h + ze > GX)
        part = hp + 0.5 * (z + ze) if self.sph else 0.5 * torch.where(out, dz, dze)
        DD = torch.where(both, d2, part)
        ok = (both | out | inn) & (DD >= GX) & (h > LAND) & (hp > LAND)
        DF = torch.where(both, d1, part).clamp_min(float(F32(1e-3)))
        DD = torch.where(ok, DD, 1.0)
        qq = 0.25 * (q + _sh(q, 0, 1) + _sh(q, -1, 0) + _sh(q, -1, 1))
        FF = self.kf * torch.sqrt(p * p + qq * qq) / DF ** MAN
        X = p - press * DD * (ze - z) + 4.0 * cor * qq
        if fric:
            X = X - FF * p
        adv = core & (d1 >= GX)
        sd = d1.clamp_min(GX)
        a, b = p * p / sd, p * qq / sd
        dw = _sh(d1, 0, -1)
        right = torch.where((_sh(d1, 0, 1) < GX) | (dze < GX), -a, _sh(a, 0, 1) - a)
        left = torch.where((dw < GX) | (dz < GX), a, a - _sh(a, 0, -1))

        def cross(s):
            gone = (_sh(dz, s, 0) < GX) | (_sh(dze, s, 0) < GX) | (_sh(d1, s, 0) < GX)
            nb = _sh(b, s, 0)
            return torch.where(gone, -b, nb - b) if s > 0 else torch.where(gone, b, b - nb)

        t = fa * torch.where(p < 0, right, left) + fc * torch.where(qq < 0, cross(1), cross(-1))
        X = torch.where(adv, X - brk * t, X)
        X = X / (1.0 + FF)
        X = torch.where(X.abs() < EPS, 0.0, X)
        return torch.where(ok, torch.minimum(torch.maximum(X, -VLIM * DD), VLIM * DD), 0.0)

    def rotate(self):
        if not self.root:  # ghost column and row
            self.z2[:, 0], self.z2[0] = self.z2[:, 1], self.z2[1]
        self.z, self.m, self.n = self.z2, self.m2, self.n2


def _edges(P, C, t, cache):
    """JNQ (t = 1) and NEWQ: the child's boundary fluxes from the parent's."""
    i0, i1, j0, j1 = C.s.corners
    R, RT = C.s.rel_size, C.s.rel_time
    wet = P.h + P.z2 > GX
    if t == 2:
        seen = P.zmax
        P.momentum()
        cache["m"], cache["n"], P.zmax = P.m2, P.n2, seen
    f = {}
    for k, a, dj, di in (("m", P.m, 0, 1), ("n", P.n, 1, 0)):
        if t > 1:
            c1 = (t - 1.0) / RT
            a = torch.where(wet & _sh(wet, dj, di), c1 * cache[k] + (1.0 - c1) * a, 0.0)
        f[k] = a
    kk = torch.arange(1, R + 1, device=P.h.device, dtype=torch.float64)

    def line(v):  # v: parent values at first-1 .. last+1 along the line
        fs, fe = 0.5 * (v[:-2] + v[1:-1]), 0.5 * (v[2:] + v[1:-1])
        c1 = (fe - fs) / (2 * R)
        return (2.0 * kk[None, :] * c1[:, None] + (fs - c1)[:, None]).reshape(-1)

    cw = C.h + C.z > GX
    for col, i in ((0, i0 - 2), (-1, i1 - 1)):
        C.m[1:, col] = torch.where(cw[1:, col], line(f["m"][j0 - 2:j1 + 1, i]), 0.0)
    for row, j in ((0, j0 - 2), (-1, j1 - 1)):
        C.n[row, 1:] = torch.where(cw[row, 1:], line(f["n"][j, i0 - 2:i1 + 1]), 0.0)


def _up(P, C):
    """JNZ: the parent's elevation from the wet child cells under it."""
    i0, i1, j0, j1 = C.s.corners
    R = C.s.rel_size
    blk = lambda a: a[1:, 1:].reshape(j1 - j0 + 1, R, i1 - i0 + 1, R)  # noqa: E731
    zc = 0.5 * (C.z + C.z2) if C.s.rel_time % 2 == 0 else C.z2
    wet = C.h + C.z2 > GX
    s, c = blk(torch.where(wet, zc, 0.0)).sum((1, 3)), blk(wet.double()).sum((1, 3))
    P.z2[j0 - 1:j1, i0 - 1:i1] = torch.where(c > R * R / 2.0, s / c.clamp_min(1.0), 0.0)


def exact(case, seed):
    cost = work(case)["flops"]
    if case["kind"] in ("batch", "source") or cost > 8e11:
        return None
    sc = _scenarios(case, seed)[0]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    layers = [_Exact(s, dev) for s in sc.layers]
    P, cache = layers[0], {}
    for _ in range(sc.steps):
        P.mass()
        for C in layers[1:]:
            for t in range(1, C.s.rel_time + 1):
                _edges(P, C, t, cache)
                C.mass()
                C.momentum()
                if t == C.s.rel_time // 2 + 1:
                    _up(P, C)
                C.rotate()
        P.momentum()
        P.rotate()
    return {f"layer{e.s.id}": {"z": e.z, "m": e.m, "n": e.n, "zmax": e.zmax, "arrival": None}
            for e in layers}
