"""Performance cases: the work a user of hemepure_amd has it do, through its
public entry points.

A case names a vessel (a pipe, a Y-bifurcation or a branching tree, given by a
few numbers), the collision and boundary selection, the storage precision and
what one pass does with the running simulation:

  fields      advance `steps` time steps, read density, velocity and wall
              shear stress back: a solver run between two outputs
  coupled     the same one step per call with the flow monitors after each: a
              program that couples to the solver every step
  checkpoint  advance, check stability, save the distributions and restart
              from them
  stress      advance, read the 17 stress components of an extraction record
  ensemble    many pipes of uneven size advanced together in a Batch
  serve       solve requests through a Server, from submission to results

listed() is the set that is tracked, draw() gives another case of the same
ranges, prepare() builds what the program holds before the call, run() is one
pass, work() the bytes and operations it cannot do without, and exact() the
same outputs from a plain 64-bit torch lattice-Boltzmann step.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import hemepure_amd as H

# D3Q19: vectors, weights and opposite directions.
C = torch.tensor([[0, 0, 0], [1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1],
                  [1, 1, 0], [-1, -1, 0], [1, -1, 0], [-1, 1, 0], [1, 0, 1], [-1, 0, -1], [1, 0, -1],
                  [-1, 0, 1], [0, 1, 1], [0, -1, -1], [0, 1, -1], [0, -1, 1]])
W = torch.tensor([1 / 3] + [1 / 18] * 6 + [1 / 36] * 12, dtype=torch.float64)
INV = [0] + [k + 1 if k % 2 else k - 1 for k in range(1, 19)]

KERNELS = {"lbgk": H.KERNEL_LBGK, "trt": H.KERNEL_TRT, "les": H.KERNEL_LES}
WALLS = {"sbb": H.WALL_SBB, "bfl": H.WALL_BFL}
TRT_LAMBDA = 3.0 / 16.0
MARGIN = 3  # solid sites around the vessel in its box
PERIOD = 2000.0  # cosine iolets, in steps


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ---- the cases --------------------------------------------------------------


def listed():
    return [
        # The straight 31k-site cylinder on which a solver is first validated: launch and latency bound.
        dict(name="cylinder-fp64", do="fields", shape="pipe", radius=10.0, length=100, narrow=0.0, kernel="lbgk",
             wall="sbb", inlet="pressure", outlet="pressure", fp32=False, steps=500),
        # The thinnest vessel of an ensemble alone, in the shifted single-precision form.
        dict(name="thin-pipe-fp32", do="fields", shape="pipe", radius=6.0, length=60, narrow=0.3, kernel="trt",
             wall="bfl", inlet="pressure", outlet="pressure", fp32=True, steps=500),
        # A small vessel inside a coupled program that looks at the flow after every step.
        dict(name="coupled-pipe-fp64", do="coupled", shape="pipe", radius=8.5, length=77, narrow=0.5, kernel="trt",
             wall="bfl", inlet="pressure", outlet="pressure", fp32=False, steps=25),
        # The 0.7M-site Y-bifurcation with a parabolic velocity inlet, both storage forms: the everyday solve.
        dict(name="bifurcation-fp64", do="fields", shape="fork", radius=24.0, length=200, seed=1, kernel="trt",
             wall="bfl", inlet="velocity", outlet="pressure", fp32=False, steps=400),
        dict(name="bifurcation-fp32", do="fields", shape="fork", radius=24.0, length=200, seed=1, kernel="trt",
             wall="bfl", inlet="velocity", outlet="pressure", fp32=True, steps=400),
        # A stenosed artery whose distributions no longer fit any cache, of an odd length.
        dict(name="artery-fp64", do="fields", shape="pipe", radius=37.3, length=501, narrow=0.5, kernel="lbgk",
             wall="bfl", inlet="pressure", outlet="pressure", fp32=False, steps=300),
        # Vessel trees with the turbulence model and Windkessel outlets: the production runs.
        dict(name="tree-fp64", do="fields", shape="tree", radius=45.0, levels=4, seed=3, kernel="les", wall="sbb",
             inlet="pressure", outlet="windkessel", fp32=False, steps=300),
        dict(name="large-tree-fp32", do="fields", shape="tree", radius=57.0, levels=5, seed=3, kernel="les",
             wall="sbb", inlet="pressure", outlet="windkessel", fp32=True, steps=300),
        # An uncertainty-quantification ensemble: uneven pipes advanced by one launch per step.
        dict(name="ensemble-fp32", do="ensemble", members=20, seed=5, fp32=True, steps=300),
        # Saving and restarting a bifurcation run.
        dict(name="checkpoint-fp64", do="checkpoint", shape="fork", radius=20.0, length=170, seed=2, kernel="lbgk",
             wall="bfl", inlet="velocity", outlet="pressure", fp32=False, steps=50),
        # An extraction record with the stress fields.
        dict(name="stress-fp32", do="stress", shape="fork", radius=20.0, length=170, seed=2, kernel="trt", wall="bfl",
             inlet="velocity", outlet="pressure", fp32=True, steps=50),
        # A handful of requests of uneven size arriving at a server together.
        dict(name="serve-fp32", do="serve", members=8, seed=9, fp32=True, steps=400),
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    do = rng.choice(["fields"] * 6 + ["coupled", "ensemble", "checkpoint", "stress", "serve"])
    if do in ("ensemble", "serve"):
        return dict(do=do, members=rng.randint(3, 20 if do == "ensemble" else 8), seed=rng.randint(1, 9999),
                    fp32=True, steps=100 * rng.randint(1, 3))
    small = do == "coupled"
    c = dict(do=do, kernel=rng.choice(["lbgk", "trt", "les"]), wall=rng.choice(["sbb", "bfl"]),
             fp32=rng.random() < 0.5)
    shape = "pipe" if small else rng.choice(["pipe", "fork", "tree"])
    if shape == "pipe":
        r = log(5.0, 12.0 if small else 40.0)
        c.update(shape=shape, radius=round(r, 2), length=int(r * rng.uniform(6.0, 14.0)) | 1,
                 narrow=round(rng.uniform(0.0, 0.7), 2), inlet=rng.choice(["pressure", "velocity"]), outlet="pressure")
    elif shape == "fork":
        r = log(7.0, 30.0)
        c.update(shape=shape, radius=round(r, 2), length=int(8 * r), seed=rng.randint(1, 9999),
                 inlet=rng.choice(["pressure", "velocity"]), outlet=rng.choice(["pressure", "windkessel"]))
    else:
        c.update(shape=shape, radius=round(log(16.0, 50.0), 2), levels=rng.randint(3, 4), seed=rng.randint(1, 9999),
                 inlet="pressure", outlet="windkessel")
    c["steps"] = rng.randint(10, 25) if small else rng.randint(20, 60) if do != "fields" else rng.randint(150, 300)
    return c


def _members(case):
    """The single-lattice cases of an ensemble or of a server's requests."""
    rng = random.Random(case["seed"])
    out = []
    for _ in range(case["members"]):
        r = rng.uniform(6.0, 18.0)
        m = dict(do="fields", shape="pipe", radius=round(r, 2), length=int(rng.uniform(60, 300)),
                 narrow=round(rng.uniform(0.0, 0.7), 2), kernel="trt", wall="bfl", inlet="pressure",
                 outlet="pressure", fp32=True, steps=case["steps"])
        if case["do"] == "serve" and rng.random() < 0.4:
            m.update(shape="fork", radius=round(rng.uniform(8.0, 14.0), 2), seed=rng.randint(1, 9999), kernel="lbgk")
            m["length"] = int(8 * m["radius"])
        out.append(m)
    return out


# ---- vessels ----------------------------------------------------------------


def _segments(case):
    """Centre lines (p0, p1, radius, children) with p in box coordinates; segment 0 starts at the inlet."""
    r = case["radius"]
    if case["shape"] == "pipe":
        return [((0.0, 0.0, 0.0), (0.0, 0.0, float(case["length"])), r, 0)]
    rng = random.Random(case["seed"])
    if case["shape"] == "fork":
        depth, taper, length = 2, 19.0 / 24.0, lambda k, rad: case["length"] * (1.0, 0.8)[k]
    else:
        depth, taper, length = case["levels"], 0.79, lambda k, rad: 3.0 * rad
    segs = []

    def grow(p, axis, rad, k):
        ln = length(k, rad)
        q = tuple(a + ln * b for a, b in zip(p, axis))
        segs.append((p, q, rad, 0 if k + 1 == depth else 2))
        if k + 1 == depth:
            return
        # two children either side of the axis, in a plane turned at random about it
        turn = rng.uniform(0.0, 2.0 * math.pi)
        ref = (1.0, 0.0, 0.0) if abs(axis[0]) < 0.9 else (0.0, 1.0, 0.0)
        e1 = np.cross(axis, ref)
        e1 /= np.linalg.norm(e1)
        side = math.cos(turn) * e1 + math.sin(turn) * np.cross(axis, e1)
        for sign in (1.0, -1.0):
            a = math.radians(rng.uniform(24.0, 40.0))
            grow(q, tuple(math.cos(a) * np.asarray(axis) + sign * math.sin(a) * side), rad * taper, k + 1)

    grow((0.0, 0.0, 0.0), (0.0, 0.0, 1.0), r, 0)
    return segs


class _Vessel:
    """A vessel voxelised: the sites in the order hemepure_amd reports them in
    (collision class, then block, then z fastest), their links, wall distances
    and normals, and the iolets (the inlet first, then the outlets)."""

    def __init__(self, case, links=True):
        dev = _device()
        segs = _segments(case)
        pts = np.array([p for s in segs for p in (np.array(s[0]), np.array(s[1]))])
        rad = np.array([s[2] for s in segs for _ in range(2)])[:, None]
        lo = np.floor((pts - rad).min(0)) - MARGIN
        hi = np.ceil((pts + rad).max(0)) + MARGIN
        lo[2] = -MARGIN - 0.5  # the inlet plane lies half-way between two layers of sites
        self.blocks = tuple(int(math.ceil((h - l + 1) / 8)) for l, h in zip(lo, hi))
        dims = tuple(8 * b for b in self.blocks)
        phi = torch.full(dims, 1e3, dtype=torch.float32, device=dev)  # signed distance, negative inside
        end = torch.full(dims, -2, dtype=torch.int8, device=dev)  # -1: inside, k: beyond iolet k's plane
        self.iolets = []
        for p0, p1, r, kids in segs:
            a, b = np.array(p0) - lo, np.array(p1) - lo
            axis = (b - a) / np.linalg.norm(b - a)
            w = [(max(0, int(min(u, v) - r - 2)), min(d, int(max(u, v) + r + 3))) for u, v, d in zip(a, b, dims)]
            box = tuple(slice(*v) for v in w)
            g = torch.meshgrid(*[torch.arange(*v, device=dev, dtype=torch.float32) for v in w], indexing="ij")
            d = [x - float(o) for x, o in zip(g, a)]
            s = sum(x * float(t) for x, t in zip(d, axis))
            ln = float(np.linalg.norm(b - a))
            sc = s.clamp(0.0, ln)
            near = torch.sqrt(sum((x - sc * float(t)) ** 2 for x, t in zip(d, axis)))
            if case["shape"] == "pipe":
                near = near - r * torch.sqrt(1.0 - case["narrow"] * torch.exp(-((s - 0.5 * ln) / (2.0 * r)) ** 2))
            else:
                near = near - r
            mark = torch.full_like(end[box], -1)
            if not self.iolets:
                mark[s < 0] = 0
                self.iolets.append((tuple(a), tuple(axis), r))
            if kids == 0:
                mark[s > ln] = len(self.iolets)
                self.iolets.append((tuple(b), tuple(-axis), r))
            closer = near < phi[box]
            phi[box] = torch.where(closer, near, phi[box])
            end[box] = torch.where(closer, mark, end[box])
        fluid = (phi < 0) & (end == -1)
        self.n = int(fluid.sum())
        if not links:
            return
        pos = fluid.nonzero()  # x, y, z with z fastest
        flat = (pos[:, 0] * dims[1] + pos[:, 1]) * dims[2] + pos[:, 2]
        fl, ph, en = fluid.reshape(-1), phi.reshape(-1), end.reshape(-1)
        here = ph[flat]
        kind = torch.zeros((self.n, 18), dtype=torch.uint8, device=dev)
        which = torch.full((self.n, 18), -1, dtype=torch.int32, device=dev)
        dist = torch.full((self.n, 18), -1.0, dtype=torch.float32, device=dev)
        for k in range(1, 19):
            to = flat + int((C[k, 0] * dims[1] + C[k, 1]) * dims[2] + C[k, 2])
            out = ~fl[to]
            io = out & (ph[to] < 0)
            kind[:, k - 1] = torch.where(io, torch.where(en[to] == 0, 2, 3), out.to(torch.uint8))
            which[:, k - 1] = torch.where(io, (en[to].int() - 1).clamp(min=0), -1)
            dist[:, k - 1] = torch.where(out, (here / (here - ph[to])).clamp(0.02, 0.98), -1.0)
            dist[:, k - 1] = torch.where(io, 0.5, dist[:, k - 1])
        wall, inl, outl = ((kind == v).any(1) for v in (H.LINK_WALL, H.LINK_INLET, H.LINK_OUTLET))
        cls = torch.where(inl, 2, torch.where(outl, 3, 0)) + torch.where(inl | outl, 2 * wall, wall)
        b, q = pos // 8, pos % 8
        block = (b[:, 0] * self.blocks[1] + b[:, 1]) * self.blocks[2] + b[:, 2]
        order = torch.argsort((cls * (int(block.max()) + 1) + block) * 512 + (q[:, 0] * 8 + q[:, 1]) * 8 + q[:, 2])
        slope = [ph[flat + st] - ph[flat - st] for st in (dims[1] * dims[2], dims[2], 1)]
        grad = torch.stack(slope, 1)
        grad = grad / grad.norm(dim=1, keepdim=True).clamp(min=1e-6)
        self.pos, self.dims, self.wall = pos[order], dims, wall[order]
        self.kind, self.which, self.dist = kind[order], which[order], dist[order]
        self.normal = torch.where(self.wall[:, None], grad[order], 0.0)

    def geometry(self):
        return H.Geometry(self.blocks, self.pos.int().cpu().numpy(), self.kind.cpu().numpy(),
                          self.which.cpu().numpy(), self.dist.cpu().numpy(),
                          self.wall.to(torch.uint8).cpu().numpy(), self.normal.cpu().numpy())


def _iolets(case, vessel, seed):
    """Per iolet what drives it, from the seed: cosine pressures, a parabolic velocity inlet or Windkessel outlets."""
    rng = random.Random(seed)
    out = []
    for k, (p, n, r) in enumerate(vessel.iolets):
        what = case["inlet"] if k == 0 else case["outlet"]
        amp = rng.uniform(1e-4, 1e-3)
        d = dict(position=p, normal=n, radius=r + 2.0, amp=amp, phase=rng.uniform(0.0, 6.0), what=what,
                 mean=1.0 + (2.0 * amp if k == 0 else 0.0), speed=rng.uniform(0.01, 0.03), area=math.pi * r * r,
                 r_c=1e-5, r_p=1e-3 * rng.uniform(0.5, 2.0), c=1e9)
        if what == "windkessel":
            d["position"] = tuple(a - 0.7 * b for a, b in zip(p, n))
        out.append(d)
    return out, rng.uniform(0.6, 0.9) if case["kernel"] != "les" else rng.uniform(0.52, 0.56)


def _desc(d):
    if d["what"] == "velocity":
        return H.iolet_desc(H.PARABOLIC, d["position"], d["normal"], radius=d["radius"], max_speed=d["speed"])
    if d["what"] == "windkessel":
        return H.iolet_desc(H.WK3, d["position"], d["normal"], radius=d["radius"], area=d["area"], r_c=d["r_c"],
                            r_p=d["r_p"], capacitance=d["c"])
    return H.iolet_desc(H.COSINE, d["position"], d["normal"], radius=d["radius"], density_mean=d["mean"],
                        density_amp=d["amp"], phase=d["phase"], period=PERIOD)


def _setup(case, seed):
    """(vessel, geometry, params, inlet and outlet descriptions) of one lattice."""
    v = _Vessel(case)
    io, tau = _iolets(case, v, seed)
    prm = H.params(kernel=KERNELS[case["kernel"]], wall_bc=WALLS[case["wall"]], tau=tau, trt_lambda=TRT_LAMBDA,
                   inlet_bc=H.IOLET_LADD if case["inlet"] == "velocity" else H.IOLET_NASH,
                   precision=H.FP32_SHIFTED if case["fp32"] else H.FP64)
    return v, v.geometry(), prm, [_desc(io[0])], [_desc(d) for d in io[1:]]


def _seeds(case, seed):
    return [seed * 1009 + k for k in range(case["members"])]


# ---- one pass ---------------------------------------------------------------


def prepare(case, seed):
    do = case["do"]
    if do == "serve":
        reqs = [_setup(m, s) for m, s in zip(_members(case), _seeds(case, seed))]
        return dict(do=do, server=H.Server(64 << 30, quantum_steps=100), steps=case["steps"],
                    requests=[r[1:] for r in reqs], walls=[r[0].wall.cpu().numpy() for r in reqs])
    if do == "ensemble":
        lats, walls = [], []
        for m, s in zip(_members(case), _seeds(case, seed)):
            v, geom, prm, ins, outs = _setup(m, s)
            lats.append(H.Lattice(geom, prm, ins, outs))
            walls.append(v.wall.cpu().numpy())
            lats[-1].init_equilibrium(1.0)
        return dict(do=do, lats=lats, walls=walls, batch=H.Batch(lats), steps=case["steps"])
    v, geom, prm, ins, outs = _setup(case, seed)
    lat = H.Lattice(geom, prm, ins, outs)
    lat.init_equilibrium(1.0)
    return dict(do=do, lat=lat, wall=v.wall.cpu().numpy(), steps=case["steps"])


def _read(fields, wall):
    """The fields of a record; only wall sites have a wall shear stress."""
    rho, u, wss = fields
    return rho, u, wss[wall]


def run(state):
    do, steps = state["do"], state["steps"]
    if do == "fields":
        state["lat"].step(steps, properties=True)
        return _read(state["lat"].fields(), state["wall"])
    if do == "coupled":
        lat, seen = state["lat"], []
        for _ in range(steps):
            lat.step(1, properties=True)
            m = lat.monitor()
            seen.append((m["rho_min"], m["rho_max"], m["u_max"], m["mass"]))
        return np.array(seen), *_read(lat.fields(), state["wall"])
    if do == "checkpoint":
        lat = state["lat"]
        lat.step(steps)
        stable = lat.stable()
        f = lat.download_f()
        lat.upload_f(f, lat.timestep())
        return f, stable
    if do == "stress":
        state["lat"].step(steps)
        return state["lat"].stress()
    if do == "ensemble":
        state["batch"].step(steps, properties=True)
        return [_read(lat.fields(), wall) for lat, wall in zip(state["lats"], state["walls"])]
    server = state["server"]
    ids = [server.submit(g, prm, ins, outs, max_steps=steps, period=100, tolerance=1e-9)
           for g, prm, ins, outs in state["requests"]]
    while any(server.advance()):
        pass
    out = [_read(server.fields(i), wall) for i, wall in zip(ids, state["walls"])]
    for i in ids:
        server.release(i)
    return out


def work(case):
    """Each step reads and writes 19 distributions of every site once; outputs are written once in 64 bits."""
    if "members" in case:
        parts = [work(m) for m in _members(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n, steps = _Vessel(case, links=False).n, case["steps"]
    out = {"checkpoint": 2 * 19, "stress": 17}.get(case["do"], 5)
    return {"bytes": n * (steps * 2 * 19 * (4 if case["fp32"] else 8) + 8 * out), "flops": n * steps * 300}


# ---- the same in 64 bits ----------------------------------------------------


def _second(v, c):
    """sum_k c_k c_k v_k as xx, xy, xz, yy, yz, zz."""
    pairs = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]
    return torch.stack([c[:, a] * c[:, b] for a, b in pairs]) @ v


class _Reference:
    """The D3Q19 step of a vessel in plain torch, 64 bits: collide, stream, wall and iolet links."""

    def __init__(self, case, seed):
        self.case, self.v = case, _Vessel(case)
        self.io, self.tau = _iolets(case, self.v, seed)
        v, dev, n = self.v, _device(), self.v.n
        self.c, self.w = C.to(dev, torch.float64), W.to(dev)
        flat = (v.pos[:, 0] * v.dims[1] + v.pos[:, 1]) * v.dims[2] + v.pos[:, 2]
        index = torch.full((v.dims[0] * v.dims[1] * v.dims[2],), -1, dtype=torch.int64, device=dev)
        index[flat] = torch.arange(n, device=dev)
        own = torch.arange(n, device=dev)
        # where each direction's value comes from: the upstream site, or the site's own opposite one
        self.src = torch.empty((19, n), dtype=torch.int64, device=dev)
        self.src[0] = own
        for j in range(1, 19):
            up = index[flat - int((C[j, 0] * v.dims[1] + C[j, 1]) * v.dims[2] + C[j, 2])]
            self.src[j] = torch.where(up >= 0, j * n + up, INV[j] * n + own)
        # per link k: its wall sites (with distances) and its iolet sites
        self.walls, self.links = [None], [None]
        ident = torch.where((v.kind >= 2).any(1), 0, -1)
        for k in range(1, 19):
            num = torch.where(v.kind[:, k - 1] == 2, 0, v.which[:, k - 1] + 1)
            ident = torch.where(v.kind[:, k - 1] >= 2, num, ident)
        for k in range(1, 19):
            s = (v.kind[:, k - 1] == 1).nonzero()[:, 0]
            both = v.kind[s, INV[k] - 1] == 1
            self.walls.append((s, v.dist[s, k - 1].double(), both))
            s = (v.kind[:, k - 1] >= 2).nonzero()[:, 0]
            self.links.append((s, ident[s]))
        t = lambda key: torch.tensor([d[key] for d in self.io], dtype=torch.float64, device=dev)  # noqa: E731
        self.normal, self.centre = t("normal"), t("position")
        self.normal = self.normal / self.normal.norm(dim=1, keepdim=True)
        self.flat_normal = self.normal.float().double()
        self.radius, self.speed, self.mean, self.amp, self.phase = (t(k) for k in ("radius", "speed", "mean", "amp", "phase"))
        self.velocity = [d["what"] == "velocity" for d in self.io]
        self.wk = {}
        for g, d in enumerate(self.io):
            if d["what"] != "windkessel":
                continue
            unit = self.c / self.c.norm(dim=1, keepdim=True).clamp(min=1e-9)
            near = int(((unit - self.normal[g]) ** 2).sum(1).argmin())
            s, of = self.links[INV[near]]
            s = s[of == g]
            around = ((v.pos - self.centre[g]).abs() <= 1.0).all(1).nonzero()[:, 0]
            coupled = len(around) > 0 and bool((s == around[0]).any())
            z = torch.zeros((), dtype=torch.float64, device=dev)
            self.wk[g] = dict(sites=s, coupled=coupled, new=z + 1.0, total=z, count=0, old=z, d=d)
        self.f = self.w[:, None].repeat(1, n)
        self.t = 1

    def densities(self):
        out = self.mean + self.amp * torch.cos(2.0 * math.pi / PERIOD * (self.t - 1) + self.phase)
        for g, s in self.wk.items():
            s["density"] = s["new"]
            s["flow"] = s["total"] * s["d"]["area"] / s["count"] if s["count"] else s["total"]
            out[g] = s["density"]
        return out

    def windkessel(self, u):
        for g, s in self.wk.items():
            if s["coupled"]:
                rc, rp, cp = s["d"]["r_c"], s["d"]["r_p"], s["d"]["c"]
                p = (rp * cp * s["density"] / 3.0 + (rc + rp) * (2.0 * s["flow"] - s["old"]) +
                     rc * rp * cp * (s["flow"] - s["old"])) / (1.0 + rp * cp)
                s["new"] = 3.0 * p
                s["old"] = s["flow"]
            s["total"] = -(u[:, s["sites"]] * self.normal[g][:, None]).sum()
            s["count"] = len(s["sites"])

    def equilibrium(self, rho, j, c, w):
        cj = c @ j
        return w[:, None] * (rho - 1.5 * (j * j).sum(0) / rho + 3.0 * cj + 4.5 * cj * cj / rho)

    def collide(self):
        f = self.f
        self.rho = f.sum(0)
        j = self.c.T @ f
        self.u = j / self.rho
        neq = f - self.equilibrium(self.rho, j, self.c, self.w)
        tau = self.tau
        if self.case["kernel"] == "trt":
            other = torch.tensor(INV, device=f.device)
            tm = 0.5 + TRT_LAMBDA / (tau - 0.5)
            opp = neq[other]
            post = f - 0.5 / tau * (neq + opp) - 0.5 / tm * (neq - opp)
        else:
            if self.case["kernel"] == "les":
                q = _second(neq, self.c)
                q = torch.sqrt(q[0] ** 2 + q[3] ** 2 + q[5] ** 2 + 2.0 * (q[1] ** 2 + q[2] ** 2 + q[4] ** 2))
                tau = 0.5 * (tau + torch.sqrt(tau * tau + 18.0 * math.sqrt(2.0) * 0.01 * q))
            post = f - neq / tau
        self.site_tau, self.post = tau, post

    def step(self):
        dens = self.densities()
        self.collide()
        post, u = self.post, self.u
        new = post.reshape(-1)[self.src.reshape(-1)].reshape(19, -1)
        for k in range(1, 19):
            j = INV[k]
            s, g = self.links[k]
            if len(s):
                if self.velocity[0]:
                    vel = g == 0
                else:
                    vel = torch.zeros_like(g, dtype=torch.bool)
                n = self.flat_normal[g].T
                rg = dens[g]
                jg = n * ((u[:, s] * n).sum(0) * rg)
                eq = self.equilibrium(rg, jg, self.c[j:j + 1], self.w[j:j + 1])[0]
                x = self.v.pos[s].double() + 0.5 * self.c[k] - self.centre[g]
                z = (x * self.normal[g]).sum(1)
                prof = 1.0 - ((x * x).sum(1) - z * z) / self.radius[g] ** 2
                wall = self.normal[g] * (self.speed[g] * prof * self.rho[s])[:, None]
                ladd = post[k, s] - 6.0 * self.w[k] * (wall @ self.c[k])
                new[j, s] = torch.where(vel, ladd, eq)
            s, q, both = self.walls[k]
            if self.case["wall"] == "bfl" and len(s):
                mixed = (post[k, s] + (2.0 * q - 1.0) * post[j, s]) / (2.0 * q)
                new[j, s] = torch.where(both | (q < 0.5), post[k, s], mixed)
        if self.case["wall"] == "bfl":
            for k in range(1, 19):
                s, q, both = self.walls[k]
                near = (q < 0.5) & ~both
                s, q = s[near], q[near]
                new[INV[k], s] = 2.0 * q * new[INV[k], s] + (1.0 - 2.0 * q) * new[k, s]
        self.windkessel(u)
        self.f_in, self.f = self.f, new
        self.t += 1

    def fields(self):
        """Density, velocity and wall shear stress of the step taken last."""
        wall = self.v.wall
        pi = -(self.site_tau - 0.5) * _second(self.post - self.f_in, self.c)
        xx, xy, xz, yy, yz, zz = pi[:, wall]
        n = self.v.normal[wall]
        n = (n / n.norm(dim=1, keepdim=True)).double().T
        sv = torch.stack([xx * n[0] + xy * n[1] + xz * n[2], xy * n[0] + yy * n[1] + yz * n[2],
                          xz * n[0] + yz * n[1] + zz * n[2]])
        wss = torch.sqrt(((sv * sv).sum(0) - (sv * n).sum(0) ** 2).clamp(min=0.0))
        return self.rho, self.u.T.contiguous(), wss

    def stress(self):
        """The stress components of the state that enters the next step."""
        self.collide()
        pi = -(self.site_tau - 0.5) * _second(self.post - self.f, self.c)
        xx, xy, xz, yy, yz, zz = pi
        p = (self.rho - 1.0) / 3.0
        ten = torch.stack([-xx - p, -xy, -xz, -yy - p, -yz, -zz - p])
        mises = torch.sqrt(0.5 * ((xx - yy) ** 2 + (yy - zz) ** 2 + (zz - xx) ** 2 + 6.0 * (xy ** 2 + yz ** 2 + xz ** 2)))
        rate = torch.sqrt(xx ** 2 + yy ** 2 + zz ** 2 + 2.0 * (xy ** 2 + yz ** 2 + xz ** 2))
        rate = rate / (-2.0 / 3.0 * self.rho) / (self.site_tau - 0.5)
        n = self.v.normal
        n = (n / n.norm(dim=1, keepdim=True).clamp(min=1e-30)).double().T
        a = ten
        tr = torch.stack([a[0] * n[0] + a[1] * n[1] + a[2] * n[2], a[1] * n[0] + a[3] * n[1] + a[4] * n[2],
                          a[2] * n[0] + a[4] * n[1] + a[5] * n[2]]) * self.v.wall
        tn = n * (tr * n).sum(0)
        return torch.cat([ten, mises[None], rate[None], tr, tr - tn, tn]).T.contiguous()


def exact(case, seed):
    do, steps = case["do"], case["steps"]
    if do in ("ensemble", "serve"):
        return [exact(m, s) for m, s in zip(_members(case), _seeds(case, seed))]
    ref, seen = _Reference(case, seed), []
    for _ in range(steps):
        ref.step()
        if do == "coupled":
            speed = ref.u.norm(dim=0).max()
            seen.append(torch.stack([ref.rho.min(), ref.rho.max(), speed, ref.rho.sum()]))
    if do == "coupled":
        return torch.stack(seen), *ref.fields()
    if do == "checkpoint":
        return ref.f.T.contiguous(), None
    return ref.stress() if do == "stress" else ref.fields()
