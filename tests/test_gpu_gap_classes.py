"""A step leaves out the list entries whose gap at the build is wider than the
particles can have closed since (gap classes, dem_device.h kReachGap). With
neigh_modify check no the rows are walked whole, so between two builds -- none
here after the first -- the two must agree to the last bit, while contacts form
out of every class. The runs end after odd and even numbers of steps."""
import numpy as np
import pytest

import pydem
import workloads as wl

pytestmark = pytest.mark.gpu

SKIN = 0.001
# shape (0, 0) lane groups, (0, 4) one lane, (5, 0) and (7, 0) the wavefront queues
SHAPES = {"lane_group": (0, 0), "one_lane": (0, 4), "compacted": (5, 0), "row_queue": (7, 0)}
# common velocity, thermal speed, number of particles that move against all others
MOTION = {"thermal": ((0.0, 0.0, 0.0), 0.25, 0), "as_one": ((0.3, 0.2, -0.5), 0.12, 0),
          "few_fast": ((0.0, 0.0, 0.0), 0.02, 40), "most_fast": ((0.0, 0.6, 0.0), 0.02, 700)}


def _system(motion, cdf):
    rng = np.random.default_rng(8)
    n = 1500
    common, thermal, against = MOTION[motion]
    L = 0.0285
    lo, hi = (0.0, 0.0, 0.0), (L, L, 2 * L)
    x = wl.lattice(n, lo, hi, 0.00285, 0.00015, rng)
    r = rng.uniform(0.001, 0.0014, n)
    v = np.asarray(common) + rng.normal(0.0, thermal, (n, 3)).clip(-2 * thermal, 2 * thermal)
    v[rng.permutation(n)[:against]] *= -1.0
    if motion == "few_fast":
        v[rng.permutation(n)[:40]] = (0.0, 0.0, 0.7)
    P = {"x": x, "v": v, "omega": rng.normal(0, 20.0, (n, 3)), "radius": r, "rmass": wl.sphere_mass(r, 2500.0),
         "type": np.ones(n, dtype=np.int32), "tag": np.arange(1, n + 1, dtype=np.int32)}
    params = {"dt": 5e-6, "skin": SKIN, "cdf": cdf, "boxlo": lo, "boxhi": hi, "periodic": (1, 1, 0),
              "grav_acc": (0.0, 0.0, -9.81), "gravity_first": 1, "rolling_cdt": 1}
    return params, wl.materials_single(rolling_friction=0.1), P, [(2, 0.0, 1)]


def _run(system, precision, shape, check, pieces):
    params, mats, P, walls = system
    params = dict(params) if check else dict(params, neigh_check=False, neigh_every=100_000)
    g = pydem.GpuSystem(params, mats, P, walls, precision=precision, max_neighbors=64)
    g.set_step_shape(*shape)
    g.run(pieces[0])
    for k in pieces[1:]:
        g.run_continue(k)
    out = g.state(), g.stats(), g.pairs()
    g.close()
    return out


def _gaps(x, r, params):
    L = np.array(params["boxhi"]) - np.array(params["boxlo"])
    d = x[:, None] - x[None]
    for k in range(2):
        d[..., k] -= L[k] * np.round(d[..., k] / L[k])
    g = np.sqrt((d ** 2).sum(-1)) - r[:, None] - r[None]
    return g[np.triu_indices(len(x), 1)]


@pytest.mark.parametrize("precision", [pydem.DEM_FP64, pydem.DEM_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("motion,cdf", [("thermal", 1.0), ("as_one", 1.0), ("few_fast", 1.0), ("most_fast", 1.0),
                                        ("thermal", 1.1)])
def test_equal_to_whole_rows(motion, cdf, shape, precision):
    system = _system(motion, cdf)
    params, _, P, _ = system
    # as far as no particle has moved half a skin, the collisions' pushes included
    share = 0.28 if motion == "most_fast" else 0.45
    steps = int(share * SKIN / (params["dt"] * np.sqrt((P["v"] ** 2).sum(1)).max())) - 3
    pieces = [steps // 3 | 1, steps // 4 & ~1, 1]
    pieces.append(steps - sum(pieces))
    print(f"[gpu] gap classes {motion} cdf {cdf} {shape}: {pieces} steps", flush=True)
    a, sa, pa = _run(system, precision, SHAPES[shape], True, pieces)
    b, sb, pb = _run(system, precision, SHAPES[shape], False, pieces)
    assert sa["nrebuilds"] == sb["nrebuilds"] == 1
    for k in ("x", "v", "omega", "f", "torque"):
        assert np.array_equal(a[k], b[k]), k
    for k in ("npairs", "ncontacts", "nwall_contacts"):
        assert sa[k] == sb[k], k
    for s, t in zip(pa, pb):
        assert np.array_equal(s, t)
    # contacts formed across wide gaps (kReachGap, in skin / 512), in thermal
    # motion across those of every class
    g0, g1 = _gaps(P["x"], P["radius"], params), _gaps(a["x"], P["radius"], params)
    first = g0[(g0 > 0) & (g1 < 0)] / SKIN * 512
    assert (first >= 88).any()
    if motion == "thermal":
        assert np.histogram(first, [0, 32, 88, 176, 1024])[0].all()
