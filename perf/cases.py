"""What is measured: the calls a user of this library makes, as cases.

A case is a scene (or a training set) with its sizes and options.  `prepare`
puts the scene on the device as a program does before its loop, `run` is one
turn of that loop: `steps` substeps, then the download of the new state, and
`exact` computes the same state with plain torch in float64.  Scenes are the
jittered lattices of the configurations in lustrine_amd/scenes.py (dam breaks
at h = 2, sand at h = 1.55), with the jitter, velocities and phases drawn from
the seed.
"""
import math

import numpy as np
import torch

from lustrine_amd import gpu as G
from lustrine_amd import learned, scenes

DT = 1.0 / 60.0


def _pbf(lattice, box, **kw):
    c = {"kind": "pbf", "nx": lattice[0], "ny": lattice[1], "nz": lattice[2], "bx": box[0], "by": box[1],
         "bz": box[2], "iterations": 4, "exact": False, "graph": True, "steps": 1, "jitter": 0.005, "speed": 0.0}
    c.update(kw)
    return c


def _sand(lattice, box, **kw):
    c = {"kind": "sand", "nx": lattice[0], "ny": lattice[1], "nz": lattice[2], "bx": box[0], "by": box[1],
         "bz": box[2], "floor": True, "graph": False, "variant": 0, "attract": False, "steps": 1, "jitter": 0.1}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest scene of an interactive program, one frame: what the calls themselves cost
        dict(_pbf((8, 8, 8), (16, 16, 16), graph=False), name="pbf_512_frame"),
        # the 32,768-particle dam break, a third of a second of simulated time between two saved states
        dict(_pbf((32, 32, 32), (64, 64, 64), steps=20), name="pbf_32k_run"),
        # a ragged scene in the reference's order of operations, for comparison with the CPU path
        dict(_pbf((47, 46, 49), (94, 92, 98), exact=True, graph=False, steps=8, jitter=0.02, speed=1.0),
             name="pbf_exact_106k"),
        # the 1,048,576-particle dam break, the configuration the benchmark quotes
        dict(_pbf((128, 64, 128), (256, 128, 256), steps=20), name="pbf_1m_run"),
        # four times as many: the neighbour lists no longer fit the last-level cache
        dict(_pbf((256, 64, 256), (512, 128, 512), steps=10), name="pbf_4m_run"),
        # many independent scenes of 4,096 to 200,000 particles per launch
        dict(_pbf((0, 0, 0), (0, 0, 0), steps=8), kind="batch", scenes=64, lo=4096, hi=200000, sizes=4,
             name="batch_64"),
        # sand and fluid falling on a voxel heightfield of static solids
        dict(_pbf((64, 64, 64), (128, 128, 128), steps=10, iterations=3), kind="mixed", hmax=16, field=11,
             name="mixed_262k"),
        # the learned warm start: features, network, three plain iterations, the bounded rerun
        dict(_pbf((128, 64, 128), (256, 128, 256), steps=10, iterations=16), kind="learned", after=3, bound=0.175,
             name="learned_1m"),
        # a level of the game: ragged sand over a solid floor with the player attracting it, one frame
        dict(_sand((41, 37, 43), (96, 80, 96), attract=True), name="sand_65k_frame"),
        # the reference's default solver on the million-particle lattice, enqueued without waiting
        dict(_sand((128, 64, 128), (256, 128, 256), floor=False, graph=True, steps=10, jitter=0.005),
             name="sand_1m_run"),
        # the reference's fluid solver with its sequential pressure sweep
        {"kind": "fluid", "nx": 32, "ny": 32, "nz": 32, "bx": 64, "by": 64, "bz": 64, "floor": True, "steps": 1,
         "name": "fluid_32k"},
        # fitting a warm-start network to recorded features
        {"kind": "fit", "rows": 131072, "epochs": 4, "batch": 4096, "name": "fit_131k"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _block(rng, n):
    """An uneven lattice of about n sites and a box some 1.5 to 2.5 times its size."""
    ny = max(2, int(round((n / rng.uniform(1.0, 4.0)) ** (1.0 / 3.0))))
    nx = max(2, int(round(math.sqrt(n / ny * rng.uniform(0.5, 2.0)))))
    nz = max(2, int(round(n / (nx * ny))))
    return (nx, ny, nz), tuple(int(math.ceil(d * rng.uniform(1.5, 2.5))) + 4 for d in (nx, ny, nz))


def draw(rng):
    kind = rng.choice(["pbf"] * 7 + ["batch"] * 2 + ["mixed"] * 3 + ["learned"] * 2 + ["sand"] * 4 + ["fluid"] * 2 + ["fit"])
    graph = rng.random() < 0.6
    if kind == "pbf":
        n = _log(rng, 400, 2000000)
        lat, box = _block(rng, n)
        exact = rng.random() < 0.25
        return _pbf(lat, box, exact=exact, graph=graph, iterations=rng.randint(1, 8),
                    steps=rng.randint(1, max(1, min(20, 8000000 // n))), jitter=rng.choice([0.005, 0.02, 0.1]),
                    speed=rng.choice([0.0, 0.5, 2.0]))
    if kind == "batch":
        return dict(_pbf((0, 0, 0), (0, 0, 0), steps=rng.randint(1, 8), graph=graph), kind="batch",
                    scenes=rng.randint(2, 40), lo=1000, hi=_log(rng, 5000, 100000), sizes=rng.randint(5, 1000))
    if kind == "mixed":
        n = _log(rng, 2000, 300000)
        lat, box = _block(rng, n)
        hmax = rng.randint(1, 16)
        return dict(_pbf(lat, (box[0], box[1] + hmax + 2, box[2]), exact=rng.random() < 0.25, graph=graph,
                         iterations=rng.randint(1, 5), steps=rng.randint(1, 10), jitter=rng.choice([0.005, 0.1])),
                    kind="mixed", hmax=hmax, field=rng.randint(12, 1000))
    if kind == "learned":
        n = _log(rng, 8000, 1000000)
        lat, box = _block(rng, n)
        return dict(_pbf(lat, box, graph=graph, iterations=rng.randint(4, 16),
                         steps=rng.randint(1, max(1, min(10, 4000000 // n)))), kind="learned", after=rng.randint(2, 4),
                    bound=rng.choice([0.175, 0.3]))
    if kind == "sand":
        n = _log(rng, 1000, 1000000)
        lat, box = _block(rng, n)
        return _sand(lat, box, floor=rng.random() < 0.7, graph=graph, variant=rng.choice([0, 0, 1]),
                     attract=rng.random() < 0.3, steps=rng.randint(1, max(1, min(10, 8000000 // n))),
                     jitter=rng.choice([0.005, 0.1, 0.2]))
    if kind == "fluid":
        lat, box = _block(rng, _log(rng, 1000, 60000))
        return {"kind": "fluid", "nx": lat[0], "ny": lat[1], "nz": lat[2], "bx": box[0], "by": box[1], "bz": box[2],
                "floor": rng.random() < 0.7, "steps": rng.randint(1, 2)}
    batch = 32 * rng.choice([8, 33, 64, 128, 200])
    return {"kind": "fit", "rows": batch * 2 + _log(rng, 5000, 250000), "epochs": rng.randint(1, 4), "batch": batch}


# ---------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _lattice(lat, origin, jitter, gen):
    """Sites of the lattice in x, y, z order with uniform jitter, on the host."""
    ax = [torch.arange(d, device="cuda", dtype=torch.float32) for d in lat]
    p = torch.stack([a.reshape(-1) for a in torch.meshgrid(*ax, indexing="ij")], 1)
    p = p + torch.tensor(origin, device="cuda", dtype=torch.float32) + 0.5
    u = torch.rand(p.shape, generator=gen, device="cuda")
    return (p + (2.0 * u - 1.0) * jitter).cpu().numpy()


def _config(case):
    return scenes.PbfConfig(name="case", lattice=(case["nx"], case["ny"], case["nz"]),
                            box=(case["bx"], case["by"], case["bz"]), iterations=case["iterations"])


def _batch(case):
    """The scenes of a batch: dam breaks with log-uniform sizes (fixed by the case)."""
    r = np.random.default_rng(case["sizes"])
    sizes = np.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]), case["scenes"]))
    return [scenes.dam_break_of_size(int(round(s)), 0, iterations=case["iterations"]) for s in sizes]


def _heightfield(case):
    """One solid per voxel below the column heights 1..hmax over the whole floor (fixed by the case)."""
    r = np.random.default_rng(case["field"])
    h = r.integers(1, case["hmax"] + 1, (case["bx"], case["bz"]))
    x, y, z = np.nonzero(np.arange(case["hmax"])[None, :, None] < h[:, None, :])
    return np.stack([x, y, z], 1).astype(np.float32) + np.float32(0.5)


def _inputs(case, seed):
    """Host arrays of the scene."""
    gen = _generator(seed)
    if case["kind"] == "fit":
        # features as a step records them: offsets and moments of order one, targets that depend on them
        x = torch.randn((case["rows"], G.FEATURES), generator=gen, device="cuda")
        w = torch.randn((G.FEATURES, 3), generator=gen, device="cuda") / math.sqrt(G.FEATURES)
        y = 0.02 * (torch.tanh(x @ w) + 0.3 * torch.randn((case["rows"], 3), generator=gen, device="cuda"))
        return {"feat": x.cpu().numpy(), "target": y.cpu().numpy()}
    if case["kind"] == "batch":
        return {"pos": np.concatenate([_lattice(s.lattice, (0.0, 0.0, 0.0), case["jitter"], gen) for s in _batch(case)])}
    lat, box = (case["nx"], case["ny"], case["nz"]), (case["bx"], case["by"], case["bz"])
    if case["kind"] in ("pbf", "learned"):
        pos = _lattice(lat, (0.0, 0.0, 0.0), case["jitter"], gen)
        vel = torch.randn((pos.shape[0], 3), generator=gen, device="cuda").cpu().numpy() * np.float32(case["speed"])
        return {"pos": pos, "vel": vel if case["speed"] else None}
    mid = tuple(float((b - d) // 2) for b, d in zip(box, lat))
    if case["kind"] == "mixed":
        pos = _lattice(lat, (mid[0], float(case["hmax"] + 1), mid[2]), case["jitter"], gen)
        ph = (torch.rand(pos.shape[0], generator=gen, device="cuda") < 0.5).to(torch.int32).cpu().numpy()
        sol = _heightfield(case)
        return {"pos": np.concatenate([pos, sol]), "phase": np.concatenate([ph, np.full(len(sol), 2, np.int32)])}
    floor = np.zeros((0, 3), np.float32)
    if case["floor"]:
        floor = scenes.lattice(case["bx"], 1, case["bz"])
    if case["kind"] == "sand":
        return {"pos": _lattice(lat, (mid[0], 1.0, mid[2]), case["jitter"], gen), "solid": floor}
    # simulate_fluid: the reference's slot layout, moving particles first, solids downward from the last slot
    sand = _lattice(lat, (0.0, 1.0, 0.0), 0.005, gen)
    n, ns = len(sand), len(floor)
    total = max(n + ns, box[0] * box[1] * box[2])
    p = np.zeros((total, 3), np.float32)
    p[:n] = sand
    p[total - ns:] = floor[::-1]
    return {"pos": p, "sand": (0, n), "solid": (total - ns, total)}


class _FluidConstants:
    """The Simulation defaults that simulate_fluid reads, for a box and particle radius 0.5."""

    def __init__(self, box):
        f = np.float32
        self.particleRadius, self.kernelFactor = 0.5, 0.5
        self.kernelRadius = float(f(4.0) * f(0.5))
        self.cubic_kernel_k = float(f(8.0 / (math.pi * self.kernelRadius ** 3)))
        self.cubic_kernel_l = float(f(48.0 / (math.pi * self.kernelRadius ** 3)))
        self.mass, self.rest_density, self.relaxation_epsilon = 5.0, 24.0, 10.0
        self.s_corr_dq, self.s_corr_k, self.s_corr_n = 0.5, 1.0, 4.0
        self.gravity = (0.0, -10.0, 0.0)
        self.domainX, self.domainY, self.domainZ = (float(b) for b in box)
        self.cell_size = self.kernelRadius
        self.gridX, self.gridY, self.gridZ = (int(f(b) / f(self.cell_size)) + 1 for b in box)


def prepare(case, seed):
    x = _inputs(case, seed)
    g = G.Gpu(0)
    s = {"case": case, "gpu": g, "steps": case.get("steps", 1)}
    kind = case["kind"]
    if kind == "fit":
        s["trainer"] = g.trainer(case["rows"])
        s["trainer"].add(x["feat"], x["target"])
    elif kind == "batch":
        b = _batch(case)
        g.pbf_batch_init(G.pbf_params(b[0], exact=case["exact"]), [c.n for c in b], [c.box for c in b], x["pos"])
        g.pbf_set_graph(case["graph"])
    elif kind in ("pbf", "learned"):
        g.pbf_init(G.pbf_params(_config(case), exact=case["exact"]), x["pos"], x["vel"])
        if kind == "learned":
            g.pbf_set_network(learned.load()[0])
            g.pbf_set_mode(True, case["after"], case["bound"])
        g.pbf_set_graph(case["graph"])
    elif kind == "mixed":
        g.mix_init(G.pbf_params(_config(case), exact=case["exact"]), G.mix_params(), x["pos"], x["phase"])
        g.pbf_set_graph(case["graph"])
    elif kind == "sand":
        n, ns = len(x["pos"]), len(x["solid"])
        index = np.arange(n + ns - 1, n - 1, -1, dtype=np.int32)
        p = G.sand_params(case["bx"], case["by"], case["bz"])
        p.ptr_solid_start = n
        g.sand_init(p, x["pos"], None, None, x["solid"] if ns else None, index if ns else None)
        g.sand_set_variant(case["variant"])
        if case["graph"]:
            g.sand_set_list_capacity(64 * n)
            g.sand_set_graph(True)
        s["player"] = np.array([case["bx"] / 2, 3.0, case["bz"] / 2], np.float32)
    else:
        c = _FluidConstants((case["bx"], case["by"], case["bz"]))
        g.fluid_init(G.fluid_params(c), x["pos"], x["pos"], np.zeros_like(x["pos"]), x["sand"], x["solid"])
    return s


def run(s):
    g, case = s["gpu"], s["case"]
    kind = case["kind"]
    if kind == "fit":
        train, val = s["trainer"].fit(epochs=case["epochs"], batch=case["batch"])
        return s["trainer"].network(), train, val
    if kind == "sand":
        for _ in range(s["steps"]):
            g.sand_step(DT, attract=case["attract"], player=s["player"])
        return g.sand_download()
    if kind == "fluid":
        for _ in range(s["steps"]):
            g.fluid_step(DT)
        return g.fluid_download()
    g.pbf_step(DT, s["steps"])
    return g.pbf_download(order=1)


def work(case):
    """Per substep each particle's position and velocity come in and go out
    (48 bytes; a static solid's position comes in), and its neighbours (33.5
    in the unit lattice within h = 2, 15.6 within 1.55) enter every solver
    pass once; the state is written once more for the caller."""
    kind = case["kind"]
    if kind == "fit":
        # two passes over a training row forward and backward: 2 x 3 x 6,272 multiply-adds
        rows = case["rows"] * case["epochs"]
        return {"bytes": rows * 35 * 4, "flops": rows * 6 * 6272}
    if kind == "batch":
        n = sum(c.n for c in _batch(case))
    else:
        n = case["nx"] * case["ny"] * case["nz"]
    steps = case["steps"]
    solids = 0
    if kind == "mixed":
        solids = len(_heightfield(case))
    elif case.get("floor"):
        solids = case["bx"] * case["bz"]
    near = 15.6 if kind == "sand" else 33.5
    if kind == "sand":
        flops = near * (8 + 4 * 10)
    elif kind == "fluid":
        flops = near * (8 + 30 + 40)
    else:
        k = case["after"] if kind == "learned" else case["iterations"]
        flops = near * (8 + k * 52 + 16) + (2 * 6272 + near * 20 if kind == "learned" else 0)
    return {"bytes": steps * (48 * n + 12 * solids) + 28 * n, "flops": steps * n * flops}


# ---------------------------------------------------------------- float64
def _cells(p, cs, dims, batch=None):
    c = (p / cs).floor().long()
    key = (c[:, 1] * dims[0] + c[:, 0]) * dims[2] + c[:, 2]
    return key if batch is None else key + batch * (dims[0] * dims[1] * dims[2])


def _pairs(p, q, h, cs, dims, pb=None, qb=None):
    """Every (i, j) with |p_i - q_j| <= h, and the stencil cell (0..26 in y, x,
    z order) j lies in; pb, qb: scene of each point of a batch."""
    nb = 1 if pb is None else int(max(pb.max(), qb.max())) + 1
    ncell = dims[0] * dims[1] * dims[2]
    order = torch.argsort(_cells(q, cs, dims, qb), stable=True)
    start = torch.searchsorted(_cells(q, cs, dims, qb)[order], torch.arange(nb * ncell + 1, device=p.device))
    c = (p / cs).floor().long()
    rows, cols, rank = [], [], []
    for r in range(27):
        d = (r // 3 % 3 - 1, r // 9 - 1, r % 3 - 1)  # x, y, z
        m = c + torch.tensor(d, device=p.device)
        ok = ((m >= 0) & (m < torch.tensor(dims, device=p.device))).all(1).nonzero()[:, 0]
        m = m[ok]
        key = (m[:, 1] * dims[0] + m[:, 0]) * dims[2] + m[:, 2]
        if pb is not None:
            key = key + pb[ok] * ncell
        cnt = start[key + 1] - start[key]
        i = ok.repeat_interleave(cnt)
        base = start[key] - (cnt.cumsum(0) - cnt)
        j = order[torch.arange(len(i), device=p.device) + base.repeat_interleave(cnt)]
        hit = ((p[i] - q[j]) ** 2).sum(1) <= h * h
        rows.append(i[hit])
        cols.append(j[hit])
        rank.append(torch.full_like(rows[-1], r))
    return torch.cat(rows), torch.cat(cols), torch.cat(rank)


def _sum(i, v, n):
    out = torch.zeros((n,) + v.shape[1:], dtype=v.dtype, device=v.device)
    return out.index_add_(0, i, v)


class _Solver:
    """Constants and passes of the position-based solver in float64."""

    def __init__(self, cfg):
        h, f = cfg.h, cfg.kernel_factor
        self.h, self.f, self.hf = h, f, h * f
        self.p6 = 315.0 / (64.0 * 3.14 * self.hf ** 9)
        self.spf = 15.0 / (3.14 * self.hf ** 6 * f)
        self.rho0, self.mass, self.eps = cfg.rest_density(), cfg.mass, cfg.epsilon
        self.k, self.n, self.c = cfg.scorr_k, cfg.scorr_n, cfg.c_xsph
        self.tq3 = (self.hf ** 2 - (f * cfg.scorr_dq) ** 2) ** 3

    def terms(self, x, i, j):
        d = x[i] - x[j]
        r2 = (d * d).sum(1)
        near = r2 <= self.h * self.h
        t3 = torch.where(near, self.hf ** 2 - self.f ** 2 * r2, 0.0) ** 3
        r = r2.sqrt()
        s = torch.where(near & (r2 > 0), self.spf * (self.hf - self.f * r) ** 2 / r, 0.0)
        return d, r2, t3, s

    def lam(self, x, i, j, own=None):
        n = len(x)
        d, r2, t3, s = self.terms(x, i, j)
        c = _sum(i, t3, n) * (self.mass * self.p6 / self.rho0) - 1.0
        a = s * s * r2 if own is None else torch.where(own[j], s * s * r2, 0.0)
        grad = _sum(i, s[:, None] * d, n)
        return -c / ((self.mass / self.rho0) ** 2 * (_sum(i, a, n) + (grad * grad).sum(1)) + self.eps), c

    def move(self, x, lam, i, j):
        d, r2, t3, s = self.terms(x, i, j)
        w = (lam[i] + lam[j] - self.k * (t3 / self.tq3) ** self.n) * s
        return _sum(i, w[:, None] * d, len(x)) * (-1.0 / self.rho0)

    def xsph(self, x, v, i, j):
        d, r2, t3, s = self.terms(x, i, j)
        return v + self.c * self.p6 * _sum(i, t3[:, None] * (v[j] - v[i]), len(x))


def _contact(pi, oi, pj, oj, moves, weight, friction, mu_s, mu_k, collision=0.8, slide=0.7):
    """The contact and friction correction of one pair within the diameter 1.
    moves: j is sand (not a solid); friction: the pair has friction."""
    ij = pi - pj
    length = ij.norm(dim=1)
    zero = length == 0
    ij = torch.where(zero[:, None], torch.tensor([0.0, 1e-5, 0.0], dtype=ij.dtype, device=ij.device), ij)
    length = torch.where(zero, 1e-5, length)
    t = (collision * weight * (length - 1.0) / length)[:, None] * ij
    m = moves[:, None]
    away = torch.where(m, pj + t, pj)
    nrm = (pi - t) - away
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    rel = ((pi - t) - oi) - torch.where(m, away - oj, 0.0)
    tang = rel - (rel * nrm).sum(1, keepdim=True) * nrm
    lt, depth = tang.norm(dim=1), t.norm(dim=1)
    ratio = torch.where(depth * mu_s > lt + 1e-9, 1.0, (mu_k * depth / (lt + 1e-9)).clamp(max=1.0))
    out = -t - torch.where(friction[:, None], slide * tang * ratio[:, None], 0.0)
    return torch.where((length <= 1.0)[:, None], out, 0.0)


def _f64(a):
    return torch.from_numpy(np.asarray(a)).to("cuda", torch.float64)


def _exact_pbf(case, x):
    """Plain, batched, mixed and learned scenes."""
    kind = case["kind"]
    dt = float(np.float32(DT))
    pos = _f64(x["pos"])
    n = len(pos)
    vel = _f64(x["vel"]) if x.get("vel") is not None else torch.zeros_like(pos)
    sid, hi = None, None
    if kind == "batch":
        b = _batch(case)
        cfg = b[0]
        cnt = torch.tensor([c.n for c in b], device="cuda")
        sid = torch.arange(len(b), device="cuda").repeat_interleave(cnt)
        hi = (_f64(np.array([c.box for c in b], np.float32)) - 0.5)[sid]
        dims = tuple(max(c.grid[a] for c in b) for a in range(3))
    else:
        cfg = _config(case)
        dims = cfg.grid
        hi = _f64(np.array(cfg.box, np.float32)) - 0.5
    sol = _Solver(cfg)
    grav = _f64(np.array(cfg.gravity, np.float32))
    lo = torch.full((3,), 0.5, dtype=torch.float64, device="cuda")
    ph = torch.from_numpy(x["phase"]).cuda() if kind == "mixed" else torch.zeros(n, dtype=torch.int32, device="cuda")
    fluid, sand, fixed = ph == 0, ph == 1, (ph == 2)[:, None]
    clamp = lambda p: torch.minimum(torch.maximum(p, lo), hi)  # noqa: E731
    if kind == "learned":
        net = learned.load()[0]
        w = torch.from_numpy(net[G.NET_PARAMS:G.NET_PARAMS + G.MLP_PARAMS].copy()).cuda()
        mats, at = [], 0
        for a, o in ((32, 64), (64, 64), (64, 3)):
            mats.append((w[at:at + a * o].reshape(a, o).bfloat16().double(), w[at + a * o:at + a * o + o].double()))
            at += a * o + o
    for _ in range(case["steps"]):
        old = pos
        cur = torch.where(fixed, pos, clamp(pos + (vel + grav * dt) * dt))
        i, j, _ = _pairs(cur, cur, sol.h, cfg.cell_size, dims, sid, sid)
        start = cur

        def solve(p, count):
            for _ in range(count):
                lam, _c = sol.lam(p, i, j, fluid if kind == "mixed" else None)
                lam = torch.where(fluid, lam, 0.0)
                step = sol.move(p, lam, i, j)
                if kind == "mixed":
                    e = (sand[i] & (i != j)).nonzero()[:, 0]
                    a, b = i[e], j[e]
                    dp = _contact(p[a], old[a], p[b], old[b], sand[b], torch.where(ph[b] == 2, 1.0, 0.5).double(),
                                  ~fluid[b], 0.6, 0.4)
                    step = torch.where(sand[:, None], _sum(a, dp, n), step)
                p = torch.where(fixed, p, clamp(p + step))
            return p

        if kind == "learned":
            d = cur[j] - cur[i]
            q = d.norm(dim=1) / sol.h
            e = i != j
            count = _sum(i[e], torch.ones_like(q[e]), n)
            slot = i[e] * 8 + (q[e] * 8).long().clamp(max=7)
            bins = _sum(slot, torch.cat([d[e] / sol.h, torch.ones_like(q[e])[:, None]], 1), n * 8).reshape(n, 8, 4)
            mean = bins[:, :, :3] / bins[:, :, 3:].clamp(min=1.0)
            near = torch.minimum(cur - lo, hi - cur).min(1).values
            per = 1.0 / count.clamp(min=1.0)
            f = torch.cat([sol.lam(cur, i, j)[1][:, None], (cur - old) / sol.h, mean.reshape(n, 24),
                           count[:, None] / 32, (_sum(i[e], q[e], n) * per)[:, None],
                           (_sum(i[e], q[e] ** 2, n) * per)[:, None], (near / sol.h).clamp(max=1.0)[:, None]], 1)
            # the network's own definition: inputs and activations are bf16 values
            f = ((f - _f64(net[:32])) * _f64(net[32:64])).bfloat16().double()
            f = torch.nn.functional.silu(f @ mats[0][0] + mats[0][1]).bfloat16().double()
            f = torch.nn.functional.silu(f @ mats[1][0] + mats[1][1]).bfloat16().double()
            cur = solve(clamp(cur + (f @ mats[2][0] + mats[2][1]) * float(net[G.NET_OUT_SCALE])), case["after"])
            if not float(sol.lam(cur, i, j)[1].max()) <= case["bound"]:
                cur = solve(start, case["iterations"])
        else:
            cur = solve(cur, case["iterations"])
        vel = (cur - old) / dt
        if kind == "mixed":
            e = (fluid[i] & fluid[j]).nonzero()[:, 0]
            vel = sol.xsph(cur, vel, i[e], j[e])
        else:
            vel = sol.xsph(cur, vel, i, j)
        pos = cur
    # a learned step's velocities follow the bf16 rounding of its features: no value of their own
    return pos, None if kind == "learned" else vel, None


def _exact_sand(case, x):
    dt = float(np.float32(DT))
    pos, solid = _f64(x["pos"]), _f64(x["solid"])
    vel = torch.zeros_like(pos)
    n, r = len(pos), 0.5
    h = float(np.float32(3.1) * np.float32(r))
    box = np.array([case["bx"], case["by"], case["bz"]], np.float32)
    dims = tuple(int(b / np.float32(h)) + 1 for b in box)
    hi = _f64(box) - r
    mu_s, mu_k = (0.95, 0.9) if case["variant"] == 0 else (0.8, 0.7)
    player = _f64(np.array([case["bx"] / 2, 3.0, case["bz"] / 2], np.float32))
    att = torch.zeros(n, dtype=torch.bool, device="cuda")
    for _ in range(case["steps"]):
        vel = vel + torch.tensor([0.0, -10.0, 0.0], dtype=torch.float64, device="cuda") * dt
        if case["attract"]:
            att = att | ((pos - player).norm(dim=1) < 1.5)
            d = player + torch.tensor([0.0, 1.5, 0.0], dtype=torch.float64, device="cuda") - pos
            vel = torch.where(att[:, None], vel + d / d.norm(dim=1, keepdim=True) * (1000.0 * r * dt / 5.0), vel)
        cur = torch.minimum((pos + vel * dt).clamp(min=r), hi)
        order = torch.argsort(_cells(cur, h, dims), stable=True)
        pos, cur, att = pos[order], cur[order], att[order]
        i, j, _ = _pairs(cur, cur, h, h, dims)
        i, j = i[i != j], j[i != j]
        a, b = (_pairs(cur, solid, h, h, dims)[:2] if len(solid) else (i[:0], i[:0]))
        for _ in range(4):
            yes, no = torch.ones_like(i, dtype=torch.bool), torch.zeros_like(a, dtype=torch.bool)
            dp = _sum(i, _contact(cur[i], pos[i], cur[j], pos[j], yes, 0.5, yes, mu_s, mu_k), n)
            if len(a):
                dp = dp + _sum(a, _contact(cur[a], pos[a], solid[b], solid[b], no, 1.0, ~no, mu_s, mu_k), n)
            cur = torch.minimum((cur + dp).clamp(min=r), hi)
        vel, pos = (cur - pos) / dt, cur
    # rows come in the last step's cell order: after several steps a particle on a cell face may
    # round to the other side and shift the rows between, which velocities do not forgive
    return pos, pos, vel if case["steps"] == 1 else None, None, None


def _exact_fluid(case, x):
    """simulate_fluid; its sequential sweep runs as levels of particles whose
    earlier neighbours are done."""
    c = _FluidConstants((case["bx"], case["by"], case["bz"]))
    h, f, dt = c.kernelRadius, c.kernelFactor, float(np.float32(0.01))
    allp = _f64(x["pos"])
    n, total = x["sand"][1], len(allp)
    pos, solid = allp[:n], allp[x["solid"][0]:]
    vel = torch.zeros_like(pos)
    hi = _f64(np.array([case["bx"], case["by"], case["bz"]], np.float32)) - c.particleRadius
    dims = (c.gridX, c.gridY, c.gridZ)

    def w(r):
        q = r * f / h
        return torch.where(q <= 0.5, c.cubic_kernel_k * (6 * q ** 3 - 6 * q ** 2 + 1),
                           c.cubic_kernel_k * 2 * (1 - q).clamp(min=0.0) ** 3)

    def grad(d):
        rl = d.norm(dim=1) * f
        q = rl / h
        s = torch.where(q <= 0.5, q * (3 * q - 2), -(1 - q) ** 2) * c.cubic_kernel_l
        s = torch.where((rl > 1e-5) & (q <= 1.0), s / (rl * h), 0.0)
        return s[:, None] * d

    w0, wq = (float(w(torch.tensor(r, dtype=torch.float64))) for r in (0.0, c.s_corr_dq))
    lam_all = torch.zeros(total, dtype=torch.float64, device="cuda")
    for _ in range(case["steps"]):
        vel = vel + torch.tensor(c.gravity, dtype=torch.float64, device="cuda") * (c.mass * dt)
        star = torch.cat([pos + vel * dt, solid])
        i, j, rank = _pairs(star[:n], star[:n], h, c.cell_size, dims)
        if len(solid):
            a, b, rs = _pairs(star[:n], solid, h, c.cell_size, dims)
            i, j, rank = torch.cat([i, a]), torch.cat([j, b + n]), torch.cat([rank, rs])
        order = torch.argsort((i * 27 + rank) * (2 * len(star)) + j)
        i, j = i[order], j[order]
        first = torch.searchsorted(i, torch.arange(n, device="cuda"))
        place = torch.arange(len(i), device="cuda") - first[i]
        rho = c.mass * (_sum(i, w((star[i] - star[j]).norm(dim=1)), n) + w0)
        gr = -(c.mass / c.rest_density) * grad(star[i] - star[j])
        norm = _sum(i, (gr * gr).sum(1), n) + (_sum(i, gr, n) ** 2).sum(1)
        lam = torch.where(norm > 0, -(rho / c.rest_density - 1.0) / (norm + c.relaxation_epsilon), 0.0)
        lam_all[:n] = lam
        other = lam_all[place]
        before = j < i
        bi, bj = i[before], j[before]
        after = torch.argsort(bj, stable=True)
        si, first_b = bi[after], torch.searchsorted(bj[after], torch.arange(n + 1, device="cuda"))
        cnt_all = torch.searchsorted(i, torch.arange(n + 1, device="cuda"))
        wait = _sum(bi, torch.ones_like(bi), n)
        ready = (wait == 0).nonzero()[:, 0]
        while len(ready):
            cnt = cnt_all[ready + 1] - cnt_all[ready]
            row = torch.arange(len(ready), device="cuda").repeat_interleave(cnt)
            e = torch.arange(len(row), device="cuda") + (cnt_all[ready] - (cnt.cumsum(0) - cnt)).repeat_interleave(cnt)
            d = star[ready][row] - star[j[e]]
            sc = -c.s_corr_k * (w(d.norm(dim=1)) / wq) ** c.s_corr_n
            p = star[ready] + _sum(row, (lam[ready][row] + other[e] + sc)[:, None] * grad(d), len(ready)) / c.rest_density
            p = torch.where(p <= c.particleRadius, 0.01, torch.where(p > hi, hi - 0.01, p))
            star[ready] = p
            cnt = first_b[ready + 1] - first_b[ready]
            e = torch.arange(int(cnt.sum()), device="cuda") + (first_b[ready] - (cnt.cumsum(0) - cnt)).repeat_interleave(cnt)
            wait[ready] = -1
            wait.index_add_(0, si[e], torch.full_like(si[e], -1))
            ready = (wait == 0).nonzero()[:, 0]
        vel, pos = (star[:n] - pos) / dt, star[:n]
    p, v = allp.clone(), torch.zeros_like(allp)
    p[:n], v[:n] = pos, vel
    return p, p, v, lam_all


def exact(case, seed):
    kind = case["kind"]
    if kind == "fit":
        return None  # its shuffles and starting weights are the library's own draws
    x = _inputs(case, seed)
    if kind == "sand":
        return _exact_sand(case, x)
    if kind == "fluid":
        return _exact_fluid(case, x)
    return _exact_pbf(case, x)
