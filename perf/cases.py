"""What a program spends its time on with this framework, as measurable cases.

Every case is one whole call sequence through the Python binding of the C ABI:
a stretch of a simulation (``run N`` and the particle state back in the
caller's order), a batch of superquadric contact points, or a stretch of the
warm-start network's training. ``listed()`` names the cases, ``draw()`` gives
others of the same ranges, ``exact()`` recomputes the sphere simulations in
64-bit torch from the contact laws and the integrator alone.

Kinds (``case["kind"]``):
  settle   polydisperse spheres r = 1.0-1.5 mm in free fall on a jittered
           3.3 mm lattice above a floor: the start of every filling
  bed      spheres at rest in contact (body-centred lattice at the mean
           diameter, about four contacts each), gravity, a floor and, with
           ``closed``, four side walls: what a filled container computes for
           most of its life; contact models hertz (cdt rolling friction),
           cohesive (hooke, no_history, sjkr) and epsd2
  drum     such a bed resting in a rotating closed cylinder of triangles
  sweep    many independent heaps of different sizes and materials on a finite
           mesh floor, advanced together (a calibration sweep)
  sqdem    superquadrics above a floor, agitated, with new contacts forming
  sqsolve  contact points of overlapping superquadric pairs
  train    the contact-point network on plain-solved pairs
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "liggghts-public_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import meshes as msh  # noqa: E402
import pydem  # noqa: E402
import superquadrics as sqm  # noqa: E402
import workloads as wl  # noqa: E402


def listed():
    return [
        # the smallest calls: one calibration-sized box stepped on its own, where launches and latency count
        {"name": "settle_4k_fp64", "kind": "settle", "n": 4000, "precision": "fp64", "steps": 500},
        # the headline workload of bench.py, in both precisions
        {"name": "settle_1m_mixed", "kind": "settle", "n": 1_000_000, "precision": "mixed", "steps": 700},
        {"name": "settle_1m_fp64", "kind": "settle", "n": 1_000_000, "precision": "fp64", "steps": 700},
        # a filled silo, full size, exact arithmetic
        {"name": "bed_1m_fp64", "kind": "bed", "n": 1_000_000, "precision": "fp64", "steps": 300, "model": "hertz",
         "closed": False},
        # a laboratory-sized fill in mixed precision, an odd particle count between walls
        {"name": "bed_150k_mixed", "kind": "bed", "n": 150_001, "precision": "mixed", "steps": 200, "model": "hertz",
         "closed": True},
        # cohesive powder: hooke, no tangential history, sjkr cohesion
        {"name": "bed_cohesive_fp64", "kind": "bed", "n": 120_000, "precision": "fp64", "steps": 300,
         "model": "cohesive", "closed": True},
        # elastic-plastic rolling friction: twice the history per contact
        {"name": "bed_epsd2_mixed", "kind": "bed", "n": 120_000, "precision": "mixed", "steps": 200,
         "model": "epsd2", "closed": False},
        # rotating drum with 2,176 moving triangles
        {"name": "drum_250k_mixed", "kind": "drum", "n": 250_000, "precision": "mixed", "steps": 200},
        # a calibration sweep of heaps, 2k-50k spheres each, replayed from captured graphs
        {"name": "sweep_48_mixed", "kind": "sweep", "instances": 48, "nmin": 2000, "nmax": 50_000,
         "precision": "mixed", "steps": 200},
        # superquadric filling
        {"name": "sqdem_50k", "kind": "sqdem", "n": 50_000, "steps": 10},
        # contact points of 100k fresh superquadric pairs
        {"name": "sqsolve_100k", "kind": "sqsolve", "n": 100_000},
        # training of the warm-start network
        {"name": "train_8k", "kind": "train", "n": 20_000, "batch": 8192, "steps": 200},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["settle", "settle", "bed", "bed", "bed", "drum", "sweep", "sqdem", "sqsolve", "train"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "settle":
        return {"kind": kind, "n": size(1000, 600_000), "precision": precision, "steps": rng.randrange(200, 801)}
    if kind == "bed":
        return {"kind": kind, "n": size(1000, 400_000), "precision": precision, "steps": rng.randrange(100, 201),
                "model": rng.choice(["hertz", "hertz", "cohesive", "epsd2"]), "closed": rng.random() < 0.5}
    if kind == "drum":
        return {"kind": kind, "n": size(10_000, 200_000), "precision": precision, "steps": rng.randrange(100, 201)}
    if kind == "sweep":
        return {"kind": kind, "instances": rng.randrange(3, 41), "nmin": 500, "nmax": size(2000, 30_000),
                "precision": precision, "steps": rng.randrange(100, 201)}
    if kind == "sqdem":
        return {"kind": kind, "n": size(1500, 40_000), "steps": rng.randrange(5, 11)}
    if kind == "sqsolve":
        return {"kind": kind, "n": size(500, 80_000)}
    return {"kind": "train", "n": size(4000, 20_000), "batch": size(500, 16_384), "steps": rng.randrange(50, 201)}


# ---------------------------------------------------------------------------
# systems
# ---------------------------------------------------------------------------
def _particles(x, v, radius, omega=None, density=2500.0):
    n = len(x)
    return {"x": np.ascontiguousarray(x), "v": v, "omega": np.zeros((n, 3)) if omega is None else omega,
            "radius": radius, "rmass": wl.sphere_mass(radius, density), "type": np.ones(n, dtype=np.int32),
            "tag": np.arange(1, n + 1, dtype=np.int32)}


def settle_system(case, seed):
    """The settling workloads: 4,000 monodisperse spheres, or polydisperse
    spheres in a column whose base grows with their number (0.3 x 0.3 m at 1M)."""
    n = case["n"]
    if n == 4000:
        return wl.settling_4k(seed=seed)
    if n == 1_000_000:
        return wl.settling_1m(seed=seed)
    rng = np.random.default_rng(seed)
    side = max(6, int(round(90 * (n / 1e6) ** (1 / 3))))
    lo, hi = (0.0, 0.0, 0.0), (side * 0.0033 + 1e-3, side * 0.0033 + 1e-3, 0.0033 * (n // side ** 2 + 12))
    r = rng.uniform(0.001, 0.0015, n)
    x = wl.lattice(n, lo, hi, 0.0033, 0.0001, rng)
    params = {"dt": 5e-6, "skin": 0.001, "cdf": 1.0, "boxlo": lo, "boxhi": hi, "periodic": (1, 1, 0),
              "grav_acc": (0.0, 0.0, -9.81), "gravity_first": 1, "rolling_cdt": 1}
    return params, wl.materials_single(rolling_friction=0.1), _particles(x, rng.normal(0.0, 0.01, (n, 3)), r), \
        [(2, 0.0, 1)]


R_BED = 0.00125


def bcc(n, side):
    """n sites of a body-centred lattice of spacing a whose nearest neighbours
    are one mean diameter less 0.2 % apart, layer by layer on side x side cells."""
    a = 2.0 * R_BED * 0.998 * 2.0 / math.sqrt(3.0)
    k = np.arange(n)
    layer, rem = k // side ** 2, k % side ** 2
    off = 0.5 * (layer % 2)
    return np.stack([(rem % side + 0.25 + off) * a, (rem // side + 0.25 + off) * a, 0.5 * layer * a], axis=1), a


def bed_system(case, seed):
    rng = np.random.default_rng(seed)
    n = case["n"]
    side = max(4, int(round((0.5 * n) ** (1 / 3))))
    x, a = bcc(n, side)
    x = x + rng.uniform(-0.004, 0.004, x.shape) * R_BED
    r = R_BED * rng.uniform(0.99, 1.01, n)
    L = side * a
    lo, hi = (0.0, 0.0, 0.0), (L, L, x[:, 2].max() * 1.05 + 8 * R_BED)
    if case["closed"]:  # side walls touch the outermost spheres
        x[:, :2] += 0.5 * (L - x[:, :2].max(0) - x[:, :2].min(0))
        walls = [(0, x[:, 0].min() - R_BED, 1), (0, x[:, 0].max() + R_BED, 1),
                 (1, x[:, 1].min() - R_BED, 1), (1, x[:, 1].max() + R_BED, 1)]
        lo, hi = (-R_BED, -R_BED, 0.0), (L + R_BED, L + R_BED, hi[2])
    else:
        walls = []
    x[:, 2] += R_BED
    walls.append((2, 0.0, 1))
    v = rng.normal(0.0, 0.01, (n, 3))
    w = rng.normal(0.0, 1.0, (n, 3))
    per = 0 if case["closed"] else 1
    params = {"dt": 5e-6, "skin": 0.001, "cdf": 1.0, "boxlo": lo, "boxhi": hi, "periodic": (per, per, 0),
              "grav_acc": (0.0, 0.0, -9.81), "gravity_first": 1, "rolling_cdt": 1}
    mats = wl.materials_single(rolling_friction=0.1)
    if case["model"] == "cohesive":
        params.update(rolling_cdt=0, normal="hooke", tangential="no_history", cohesion="sjkr")
        mats.update(cohesion_energy_density=[[2e4]], characteristic_velocity=1.0)
    elif case["model"] == "epsd2":
        params.update(rolling_cdt=0, rolling_epsd2=1)
    return params, mats, _particles(x, v, r, w), walls


DRUM_AZ, DRUM_AX = 64, 16


def drum_system(case, seed):
    """The lower half of a 64-sided drum filled with a bed whose outermost
    spheres touch the mantle and the caps; radius and length grow with n."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    # half the cylinder (radius R, length 0.7 R) holds n spheres of a bcc bed
    a = 2.0 * R_BED * 0.998 * 2.0 / math.sqrt(3.0)
    R = (n * a ** 3 / 2.0 / (0.5 * math.pi * 0.7)) ** (1 / 3) + 2.0 * R_BED
    ly = max(4, int(round(0.7 * R / a)))  # cells along the axis
    # layers of the lattice along y so that both end layers touch their caps
    nyl = 2 * ly + 1
    length = (nyl - 1) * 0.5 * a + 2.0 * R_BED
    m = int(R / a) + 2
    X, K, Z = np.meshgrid(np.arange(-m, m + 1), np.arange(nyl), np.arange(-m, m + 1), indexing="ij")
    off = 0.5 * (K % 2)
    pts = np.stack([((X + off) * a).ravel(), (K * 0.5 * a - 0.5 * (nyl - 1) * 0.5 * a).ravel(),
                    ((Z + off) * a).ravel()], axis=1)
    th = 2.0 * math.pi * (np.arange(DRUM_AZ) + 0.5) / DRUM_AZ
    apothem = R * math.cos(math.pi / DRUM_AZ)
    d = apothem - np.max(pts[:, 0:1] * np.cos(th) + pts[:, 2:3] * np.sin(th), axis=1)  # to the nearest facet
    pts = pts[d >= 0.995 * R_BED]
    pts = pts[np.lexsort((pts[:, 0], pts[:, 1], pts[:, 2]))][:n]
    n = len(pts)
    x = pts + rng.uniform(-0.004, 0.004, pts.shape) * R_BED
    r = R_BED * rng.uniform(0.99, 1.01, n)
    b = (R * 1.05, 0.5 * length * 1.2, R * 1.05)
    params = {"dt": 5e-6, "skin": 0.0005, "cdf": 1.0, "boxlo": tuple(-t for t in b), "boxhi": b,
              "periodic": (0, 0, 0), "grav_acc": (0.0, 0.0, -9.81), "gravity_first": 1, "rolling_cdt": 0}
    meshes = [(msh.drum(R, length, DRUM_AZ, DRUM_AX), 2, None, ((0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 2.0))]
    P = _particles(x, rng.normal(0.0, 0.01, (n, 3)), r)
    return params, wl.materials_two(), P, [], meshes, (R, length)


def sweep_system(case, seed):
    """Heaps as workloads.heap_sweep draws them, lowered onto the floor and
    set in motion, so that floor and pair contacts form from the first steps."""
    # sizes evenly spread over the logarithm of their range
    counts = np.exp(np.linspace(math.log(case["nmin"]), math.log(case["nmax"]), case["instances"])).round()
    params, base, P, walls, meshes, counts, imats = wl.heap_sweep(
        seed=seed, ninst=case["instances"], counts=counts.astype(np.int64))
    rng = np.random.default_rng(seed + 1)
    a = 2.2 * 0.0015
    P["x"][:, 2] -= 0.25 * a
    P["v"] = rng.normal(0.0, 0.1, P["x"].shape)
    P["v"][:, 2] -= 0.1
    return params, base, P, walls, meshes, counts, imats


def sqdem_system(case, seed):
    """The superquadric filling of bench.py (agitated start), its layer lattice
    drawn together to 0.72 so that about one particle in four touches another."""
    n, s = case["n"], 0.72
    base = max(0.045, 0.2 * (n / 200_000) ** (1 / 3))
    params, mats, P, walls = wl.superquadric_settling(seed, n, base=(base, base), gap=0.0003)
    rng = np.random.default_rng(seed + 1)
    P["x"] = P["x"] * s
    P["x"][:, 2] += 0.001
    params["boxhi"] = [base * s, base * s, params["boxhi"][2]]
    P["v"] = rng.normal(0.0, 0.3, (n, 3))
    P["omega"] = rng.normal(0.0, 30.0, (n, 3))
    return params, mats, P, walls


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _touched(shape, dtype=np.float64):
    a = np.empty(shape, dtype=dtype)
    a.fill(0)
    return a


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "steps": case.get("steps", 0)}
    if kind in ("settle", "bed", "drum", "sweep"):
        prec = pydem.DEM_MIXED if case["precision"] == "mixed" else pydem.DEM_FP64
        if kind == "settle":
            params, mats, P, walls = settle_system(case, seed)
            g = pydem.GpuSystem(params, mats, P, walls, precision=prec)
        elif kind == "bed":
            params, mats, P, walls = bed_system(case, seed)
            g = pydem.GpuSystem(params, mats, P, walls, precision=prec)
        elif kind == "drum":
            params, mats, P, walls, meshes, _ = drum_system(case, seed)
            g = pydem.GpuSystem(params, mats, P, walls, precision=prec, meshes=meshes)
        else:
            params, base, P, walls, meshes, counts, imats = sweep_system(case, seed)
            g = pydem.GpuSystem(params, base, P, walls, precision=prec, meshes=meshes, instances=counts,
                                instance_materials=imats)
            g.set_graph_capture(True)
        st["g"] = g
        # mixed precision hands out the state it advances; 64-bit runs the last forces too (see tolerance())
        names = ("x", "v", "omega") if prec == pydem.DEM_MIXED else ("x", "v", "omega", "f", "torque")
        st["out"] = {k: _touched((len(P["x"]), 3)) for k in names}
    elif kind == "sqdem":
        params, mats, P, walls = sqdem_system(case, seed)
        g = pydem.SqDemSystem(params, mats, P, walls)
        n = len(P["x"])
        st["g"] = g
        st["out"] = {k: _touched((n, 3)) for k in ("x", "v", "omega", "angmom", "f", "torque")}
        st["out"]["quat"] = _touched((n, 4))
    else:
        A, B = sqm.overlapping_pairs(seed, case["n"])
        s = pydem.SqSolver()
        s.set_pairs(A, B)
        st["s"] = s
        if kind == "train":
            s.solve(pydem.DEM_SQ_FRESH)  # the training targets
            s.net_init(seed=seed)
            st["batch"] = case["batch"]
    return st


def run(state):
    """One pass: the simulation goes on from where it is, as a program's next
    ``run N`` does, and the state comes back in the caller's arrays."""
    kind = state["kind"]
    dp = pydem._dp
    if kind == "sqsolve":
        r = state["s"].solve(pydem.DEM_SQ_FRESH)
        return {k: r[k] for k in ("point", "fi", "fj", "iters", "flags")}
    if kind == "train":
        curve, _ = state["s"].net_train(steps=state["steps"], batch=state["batch"], lr=2e-3, seed=7)
        return {"loss": curve, "params": state["s"].net_params()}
    g, o = state["g"], state["out"]
    g.run(state["steps"])
    if kind == "sqdem":
        g._check(g.lib.dem_sqdem_get_state(g.h, dp(o["x"]), dp(o["v"]), dp(o["omega"]), dp(o["angmom"]),
                                           dp(o["quat"]), dp(o["f"]), dp(o["torque"])))
    else:
        g._check(g.lib.dem_get_state(g.h, dp(o["x"]), dp(o["v"]), dp(o["omega"]), *(
            dp(o[k]) if k in o else None for k in ("f", "torque"))))
    return o


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes and flops of one pass. Spheres, per step and particle: position,
    radius, velocity, mass, angular velocity, displacement reference and list
    length read, position, velocity and angular velocity written; 4 bytes for
    each half-list pair; the history read and written and about 250 flops for
    each contact; then the state handed out. Superquadrics: about
    2,000 flops for each Newton iteration. Network: its products."""
    kind = case["kind"]
    if kind in ("settle", "bed", "drum", "sweep"):
        mixed = case["precision"] == "mixed"
        if kind == "sweep":
            # the mean of the log-uniform sizes
            lo, hi = case["nmin"], case["nmax"]
            n = case["instances"] * (hi - lo) / math.log(hi / lo)
        else:
            n = case["n"]
        per = 32 + 32 + (16 if mixed else 32) + 24 + 4 + 48 + (12 if mixed else 24)
        pairs, contacts = {"settle": (2.3, 0.0), "bed": (6.5, 2.0), "drum": (6.5, 2.0), "sweep": (3.0, 0.2)}[kind]
        hist = 0 if case.get("model") == "cohesive" else (12 if mixed else 24) * (
            2 if case.get("model") == "epsd2" else 1)
        step = n * (per + 4 * pairs + 2 * hist * contacts)
        return {"bytes": step * case["steps"] + (72 if mixed else 120) * n,
                "flops": n * (60 + 10 * pairs + 250 * contacts) * case["steps"]}
    if kind == "sqdem":
        n = case["n"]
        return {"bytes": n * case["steps"] * (400 + 8 * 240) + 176 * n,
                "flops": n * case["steps"] * (600 + 0.2 * 3 * 2000)}
    if kind == "sqsolve":
        return {"bytes": case["n"] * (192 + 48), "flops": case["n"] * 34.5 * 2000}
    return {"bytes": case["steps"] * case["batch"] * (21 * 4 + 8), "flops": case["steps"] * case["batch"] * 30208}


def tolerance(case):
    """Set from runs whose start was changed by one unit in the last place: four
    times what came out. Contacts pass a rounding difference on from step to
    step. In mixed precision the contact law rounds to 32 bits, and where two
    spheres hardly turn against each other the direction of their rolling
    torque follows the sign of that rounding, so a single particle's torque
    has no stable value (differences of several times the mean); the state it
    drives has."""
    kind = case["kind"]
    if kind == "train":  # bf16 products, 32-bit sums, and the Adam steps that pass a difference on
        return {"rel": 1e-2, "max": 0.5}
    if kind == "sqsolve":  # a solve passes rounding on through its iterations
        return {"rel": 1e-8, "max": 1e-6, "differ": 0.01}
    if kind == "sqdem":
        return {"rel": 1e-9, "max": 1e-6}
    if case["precision"] == "mixed":
        return {"rel": 2e-3, "max": 0.8}
    return {"rel": 1e-7, "max": 1e-4}


# ---------------------------------------------------------------------------
# the sphere simulations in 64 bits
# ---------------------------------------------------------------------------
class _Spheres:
    """Spheres with pair, plane and drum contacts, in float64 torch: the list
    is built with the skin, rebuilt when a particle (or mesh node) moved half
    of it, and a contact's history survives a build only while it touches."""

    def __init__(self, params, P, walls, device, inst=None, mat=None, drum=None):
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=device)  # noqa: E731
        self.p, self.dev, self.walls, self.drum = params, device, walls, drum
        self.x, self.v, self.w = t(P["x"]), t(P["v"]), t(P["omega"])
        self.r, self.m = t(P["radius"]), t(P["rmass"])
        self.inst = None if inst is None else torch.as_tensor(inst, device=device)
        self.mat = mat  # mat(index of particles, wall or not) -> dict of constants or tensors
        self.lo, self.hi = t(params["boxlo"]), t(params["boxhi"])
        self.per = params["periodic"]
        self.pairs = None
        self.wsh = [torch.zeros_like(self.x) for _ in walls]
        self.wrh = [torch.zeros_like(self.x) for _ in walls]
        self.wtouch = [torch.zeros(len(self.x), dtype=torch.bool, device=device) for _ in walls]
        self.step = 0
        if drum:
            self.dsh = torch.zeros(len(self.x), DRUM_AZ + 2, 3, dtype=torch.float64, device=device)
            self.dtouch = torch.zeros(len(self.x), DRUM_AZ + 2, dtype=torch.bool, device=device)

    def build(self):
        x, dev = self.x, self.dev
        for d in range(3):
            if self.per[d]:
                L = self.hi[d] - self.lo[d]
                x[:, d] = torch.where(x[:, d] < self.lo[d], x[:, d] + L, x[:, d])
                x[:, d] = torch.where(x[:, d] >= self.hi[d], x[:, d] - L, x[:, d])
        skin = self.p["skin"]
        cut = float(2.0 * self.r.max() + skin)
        nc = [max(1, int(float(self.hi[d] - self.lo[d]) / cut)) for d in range(3)]
        nc = [1 if (self.per[d] and nc[d] < 3) else nc[d] for d in range(3)]
        c = [((x[:, d] - self.lo[d]) / (self.hi[d] - self.lo[d]) * nc[d]).floor().long().clamp(0, nc[d] - 1)
             for d in range(3)]
        ninst = 1 if self.inst is None else int(self.inst.max()) + 1
        base = 0 if self.inst is None else self.inst.long() * (nc[0] * nc[1] * nc[2])
        cell = (c[2] * nc[1] + c[1]) * nc[0] + c[0] + base
        order = torch.argsort(cell)
        count = torch.bincount(cell, minlength=ninst * nc[0] * nc[1] * nc[2])
        start = torch.cumsum(count, 0) - count
        I, J = [], []
        offs = {d: ([0] if nc[d] == 1 else [-1, 0, 1]) for d in range(3)}
        me = torch.arange(len(x), device=dev)
        for oz in offs[2]:
            for oy in offs[1]:
                for ox in offs[0]:
                    q, ok = [], torch.ones(len(x), dtype=torch.bool, device=dev)
                    for d, o in ((0, ox), (1, oy), (2, oz)):
                        e = c[d] + o
                        if self.per[d]:
                            e = e % nc[d]
                        else:
                            ok &= (e >= 0) & (e < nc[d])
                        q.append(e)
                    i = me[ok]
                    cc = ((q[2] * nc[1] + q[1]) * nc[0] + q[0] + base)[ok]
                    k = count[cc]
                    ii = torch.repeat_interleave(i, k)
                    first = torch.repeat_interleave(start[cc] - (torch.cumsum(k, 0) - k), k)
                    jj = order[first + torch.arange(len(ii), device=dev)]
                    keep = ii < jj
                    ii, jj = ii[keep], jj[keep]
                    d2 = self.delta(ii, jj).square().sum(1)
                    near = d2 <= (self.r[ii] + self.r[jj] + skin) ** 2
                    I.append(ii[near])
                    J.append(jj[near])
        i, j = torch.cat(I), torch.cat(J)
        n = len(x)
        key, perm = torch.sort(i * n + j)
        i, j = i[perm], j[perm]
        sh = torch.zeros(len(i), 3, dtype=torch.float64, device=dev)
        rh = torch.zeros_like(sh)
        if self.pairs is not None:
            okey, osh, orh, oflag = self.key, self.sh, self.rh, self.flag
            at = torch.searchsorted(okey, key).clamp(max=max(len(okey) - 1, 0))
            if len(okey):
                touch = self.delta(i, j).square().sum(1) < (self.r[i] + self.r[j]) ** 2
                same = (okey[at] == key) & oflag[at] & touch
                sh[same], rh[same] = osh[at[same]], orh[at[same]]
                flag = same
            else:
                flag = torch.zeros(len(i), dtype=torch.bool, device=dev)
        else:
            flag = torch.zeros(len(i), dtype=torch.bool, device=dev)
        self.pairs, self.key, self.sh, self.rh, self.flag = (i, j), key, sh, rh, flag
        self.xhold = x.clone()
        self.angle_hold = self.step

    def delta(self, i, j):
        d = self.x[i] - self.x[j]
        for k in range(3):
            if self.per[k]:
                L = self.hi[k] - self.lo[k]
                d[:, k] = torch.where(d[:, k] > 0.5 * L, d[:, k] - L,
                                      torch.where(d[:, k] < -0.5 * L, d[:, k] + L, d[:, k]))
        return d

    def law(self, wall, en, dl, rinv, deltan, deltan_in, ri, rj, meff, vr, wi, wj, mat, sh, rh, update, acont):
        """Force on i and the torques of one batch of contacts; sh and rh are updated in place."""
        p = self.p
        dot = lambda a, b: (a * b).sum(1, keepdim=True)  # noqa: E731
        c1 = lambda t: t[:, None] if torch.is_tensor(t) and t.dim() == 1 else t  # noqa: E731
        deltan, deltan_in, ri, rinv, meff = map(c1, (deltan, deltan_in, ri, rinv, meff))
        Y, G, beta, loge, mu, mur = (c1(mat[k]) for k in ("Y", "G", "beta", "loge", "mu", "mur"))
        vn = dot(vr, en)
        vt = vr - vn * en
        if wall:
            cri = ri - 0.5 * deltan_in
            wr = cri * wi * rinv
            reff = ri
        else:
            rj = c1(rj)
            cri, crj = ri - 0.5 * deltan, rj - 0.5 * deltan
            wr = (cri * wi + crj * wj) * rinv
            reff = ri * rj / (ri + rj)
        vtr = vt - torch.stack(
            (dl[:, 2] * wr[:, 1] - dl[:, 1] * wr[:, 2], dl[:, 0] * wr[:, 2] - dl[:, 2] * wr[:, 0],
             dl[:, 1] * wr[:, 0] - dl[:, 0] * wr[:, 1]), 1)
        if p.get("normal") == "hooke":
            sq = torch.sqrt(reff)
            kn = 16.0 / 15.0 * sq * Y * (15.0 * meff * mat["cv"] ** 2 / (16.0 * sq * Y)) ** 0.2
            kt = kn
            gn = torch.sqrt(4.0 * meff * kn * loge ** 2 / (loge ** 2 + math.pi ** 2))
            gt = gn
        else:
            sq = torch.sqrt(reff * deltan)
            kn = 4.0 / 3.0 * Y * sq
            kt = 8.0 * G * sq
            s56 = math.sqrt(5.0 / 6.0)
            gn = -2.0 * s56 * beta * torch.sqrt(2.0 * Y * sq * meff)
            gt = -2.0 * s56 * beta * torch.sqrt(kt * meff)
        Fn = -gn * vn + kn * deltan
        F = Fn * en
        if p.get("cohesion") == "sjkr":
            F = F - mat["ced"] * c1(acont) * en
        cap = mu * Fn.abs()
        if p.get("tangential") == "no_history":
            vrel = torch.sqrt(dot(vtr, vtr))
            Ft = -torch.where(cap < gt * vrel, cap / vrel, gt * torch.ones_like(cap)) * vtr
        else:
            if update:
                sh = sh + vtr * p["dt"]
                sh = sh - dot(sh, en) * en
            mag = torch.sqrt(dot(sh, sh))
            slip = kt * mag > cap
            Fs = -kt * sh
            ratio = torch.where(slip, cap / (kt * mag), torch.ones_like(cap))
            Ft = torch.where(slip, Fs * ratio, Fs - gt * vtr)
            if update:
                sh = torch.where(slip, -Ft / kt, sh)
        F = F + Ft
        tor = torch.linalg.cross(en, Ft)
        Ti = -cri * tor
        Tj = None if wall else -crj * tor
        if p.get("rolling_epsd2"):
            ww = wr if wall else wi - wj
            ww = ww - dot(ww, en) * en
            rt = rh + p["dt"] * kt * reff * reff * ww
            rmag = torch.sqrt(dot(rt, rt))
            rmax = Fn.abs() * reff * mur
            rt = torch.where(rmag > rmax, rt * (rmax / rmag), rt)
            if update:
                rh = rt
            Ti = Ti - rt
            Tj = None if wall else Tj + rt
        elif p.get("rolling_cdt"):
            ww = wr if wall else wi - wj
            mag = torch.sqrt(dot(ww, ww))
            rt = torch.where(mag > 0, mur * kn * deltan * reff * ww / mag, torch.zeros_like(ww))
            rt = rt - dot(rt, en) * en
            Ti = Ti - rt
            Tj = None if wall else Tj + rt
        return F, Ti, Tj, sh, rh

    def forces(self, update):
        n = len(self.x)
        F = torch.zeros_like(self.x)
        T = torch.zeros_like(self.x)
        F += self.m[:, None] * torch.tensor(self.p["grav_acc"], dtype=torch.float64, device=self.dev)
        i, j = self.pairs
        d = self.delta(i, j)
        rsq = d.square().sum(1)
        rs = self.r[i] + self.r[j]
        t = torch.nonzero(rsq < rs * rs)[:, 0]
        if len(t):
            it, jt, dt_, r = i[t], j[t], d[t], torch.sqrt(rsq[t])
            en = dt_ / r[:, None]
            ri, rj = self.r[it], self.r[jt]
            meff = self.m[it] * self.m[jt] / (self.m[it] + self.m[jt])
            ac = -math.pi / 4 * (r - ri - rj) * (r + ri - rj) * (r - ri + rj) * (r + ri + rj) / (r * r)
            sh = self.sh[t] * self.flag[t][:, None]
            rh = self.rh[t] * self.flag[t][:, None]
            dl = ri + rj - r
            f, ti, tj, sh, rh = self.law(False, en, dt_, 1.0 / r, dl, dl, ri, rj, meff, self.v[it] - self.v[jt],
                                         self.w[it], self.w[jt], self.mat(it, False), sh, rh, update, ac)
            self.sh[t], self.rh[t] = sh, rh
            self.flag[t] = True
            F.index_add_(0, it, f)
            F.index_add_(0, jt, -f)
            T.index_add_(0, it, ti)
            T.index_add_(0, jt, tj)
        for k, wall in enumerate(self.walls):
            ax, pos = wall[0], wall[1]
            dist = self.x[:, ax] - pos
            touch = dist.abs() - self.r <= 0
            q = torch.nonzero(touch)[:, 0]
            if len(q):
                gap = dist[q].abs()
                en = torch.zeros(len(q), 3, dtype=torch.float64, device=self.dev)
                en[:, ax] = torch.sign(dist[q])
                self._wall(q, gap, en, torch.zeros_like(en), self.wsh[k], self.wrh[k], self.wtouch[k], update, F, T)
            self.wtouch[k] = touch
        if self.drum:
            self._drum(update, F, T)
        self.F, self.T = F, T
        assert len(F) == n

    def _wall(self, q, gap, en, vw, shs, rhs, touched, update, F, T):
        """Contacts of particles q with a wall at distance gap along -en."""
        ri = self.r[q]
        sh = shs[q] * touched[q][:, None]
        rh = rhs[q] * touched[q][:, None]
        dn = ri - gap
        f, ti, _, sh, rh = self.law(True, en, en * gap[:, None], 1.0 / gap, dn, dn, ri, None, self.m[q],
                                    self.v[q] - vw, self.w[q], None, self.mat(q, True), sh, rh, update,
                                    (ri * ri - gap * gap) * math.pi)
        shs[q], rhs[q] = sh, rh
        F.index_add_(0, q, f)
        T.index_add_(0, q, ti)

    def _drum(self, update, F, T):
        R, length, om = self.drum
        ang = om * self.p["dt"] * self.step
        ap = R * math.cos(math.pi / DRUM_AZ)
        half = R * math.sin(math.pi / DRUM_AZ)
        moving = 0.0 if self.step == 0 else 1.0
        now = torch.zeros_like(self.dtouch)
        # only particles near the mantle or a cap can touch
        rad = torch.sqrt(self.x[:, 0] ** 2 + self.x[:, 2] ** 2)
        near = torch.nonzero(rad > ap - 1.5 * self.r.max())[:, 0]
        for k in range(DRUM_AZ + 2):
            if k < DRUM_AZ:
                # rotation about +y by ang takes the angle th (from x towards z) to th - ang
                th = 2.0 * math.pi * (k + 0.5) / DRUM_AZ - ang
                nx, nz = math.cos(th), math.sin(th)
                xs, zs = self.x[near, 0], self.x[near, 2]
                gap = ap - (xs * nx + zs * nz)
                along = -xs * nz + zs * nx
                hit = (gap <= self.r[near]) & (along.abs() <= half)
                q, g = near[hit], gap[hit]
                en = torch.zeros(len(q), 3, dtype=torch.float64, device=self.dev)
                en[:, 0], en[:, 2] = -nx, -nz
            else:
                s = -1.0 if k == DRUM_AZ else 1.0
                gap = 0.5 * length - s * self.x[:, 1]
                q = torch.nonzero(gap <= self.r)[:, 0]
                g = gap[q]
                en = torch.zeros(len(q), 3, dtype=torch.float64, device=self.dev)
                en[:, 1] = -s
            if len(q):
                cp = self.x[q] - en * g[:, None]
                vw = torch.zeros_like(cp)
                vw[:, 0], vw[:, 2] = om * cp[:, 2] * moving, -om * cp[:, 0] * moving
                shs = self.dsh[:, k]
                self._wall(q, g, en, vw, shs, torch.zeros_like(shs), self.dtouch[:, k], update, F, T)
                now[q, k] = True
        self.dtouch = now

    def run(self, steps):
        dt = self.p["dt"]
        dtf = 0.5 * dt
        self.build()
        self.forces(False)
        force_build = False
        for _ in range(steps):
            self.step += 1
            self.v += dtf * self.F / self.m[:, None]
            self.x += dt * self.v
            rot = (dtf / 0.4 / (self.r * self.r * self.m))[:, None]
            self.w += rot * self.T
            lim = 0.25 * self.p["skin"] ** 2
            moved = bool(((self.x - self.xhold).square().sum(1) > lim).any())
            if moved or force_build:
                self.build()
            force_build = False
            if self.drum:
                R, _, om = self.drum
                # a mesh node half a skin away from where the last build saw it asks for a build at the next step
                if (2.0 * R * math.sin(0.5 * om * dt * (self.step - self.angle_hold))) ** 2 > lim:
                    force_build = True
            self.forces(True)
            self.v += dtf * self.F / self.m[:, None]
            self.w += rot * self.T
        return {"x": self.x, "v": self.v, "omega": self.w, "f": self.F, "torque": self.T}


def _mixed(mats, a, b):
    """Effective constants of types a and b (0-based)."""
    Y, nu = mats["youngs"], mats["poisson"]
    e, mu = mats["restitution"][a][b], mats["friction"][a][b]
    le = math.log(e)
    return {"Y": 1.0 / ((1 - nu[a] ** 2) / Y[a] + (1 - nu[b] ** 2) / Y[b]),
            "G": 1.0 / (2 * (2 - nu[a]) * (1 + nu[a]) / Y[a] + 2 * (2 - nu[b]) * (1 + nu[b]) / Y[b]),
            "beta": le / math.sqrt(le * le + math.pi ** 2), "loge": le, "mu": mu,
            "mur": mats["rolling_friction"][a][b] if "rolling_friction" in mats else 0.0,
            "cv": mats.get("characteristic_velocity", 0.0),
            "ced": mats["cohesion_energy_density"][a][b] if "cohesion_energy_density" in mats else 0.0}


def exact(case, seed):
    """The sphere simulations in 64 bits. Superquadric results have no such
    value: a contact point is by definition where the Newton iteration stops
    (within its merit tolerance, about 1e-8 m, of the exact one), and the
    network is trained on those points."""
    if case["kind"] not in ("settle", "bed", "drum", "sweep"):
        return None
    out = _exact(case, seed)
    if case["precision"] == "mixed":
        out["f"] = out["torque"] = None
    return {k: t if t is None else t.cpu().numpy() for k, t in out.items()}


def _exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "sweep":
        params, _, P, _, _, counts, imats = sweep_system(case, seed)
        inst = np.repeat(np.arange(len(counts)), counts)
        table = {}
        for k in ("Y", "G", "beta", "loge", "mu", "mur"):
            table[k] = torch.tensor([_mixed(m, 0, 0)[k] for m in imats], dtype=torch.float64, device=dev)
        inst_t = torch.as_tensor(inst, device=dev)

        def mat(q, wall):
            return {k: v[inst_t[q]] for k, v in table.items()}
        s = _Spheres(params, P, [(2, 0.0, 2)], dev, inst=inst, mat=mat)
        return s.run(case["steps"])
    if kind == "drum":
        params, mats, P, walls, _, (R, length) = drum_system(case, seed)
        s = _Spheres(params, P, walls, dev, mat=lambda q, wall: _mixed(mats, 0, 1 if wall else 0),
                     drum=(R, length, math.pi))
        return s.run(case["steps"])
    params, mats, P, walls = settle_system(case, seed) if kind == "settle" else bed_system(case, seed)
    s = _Spheres(params, P, walls, dev, mat=lambda q, wall: _mixed(mats, 0, 0))
    return s.run(case["steps"])
