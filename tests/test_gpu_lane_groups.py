"""Small systems step each particle with a group of lanes (dem_kernels.hip,
step_group). The contributions are summed in the order of the one-lane shape,
so the two give the same bits; the one-lane shape is asked for through its
persistent grid (dem_set_step_shape 0, 4). The rows hold more than 16 and more
than 32 entries where the skin is wide, and the particle counts leave a partial
block and a partial last group of blocks per XCD."""
import numpy as np
import pytest

import meshes as msh
import pydem
import workloads as wl

pytestmark = pytest.mark.gpu

SIBLING = {"normal": "hooke", "tangential": "no_history", "cohesion": "sjkr", "rolling_cdt": 0}
EPSD2 = {"rolling_epsd2": 1, "rolling_cdt": 0}

CASES = {
    "one": (1, {}, False),
    "partial_group": (7, {}, False),
    "whole_block": (16, {}, False),
    "block_and_one": (17, {}, False),
    "long_rows": (1025, {"skin": 0.0012}, False),
    "longer_rows": (900, {"skin": 0.0033}, False),
    "every_third_step": (1025, {"neigh_every": 3, "skin": 0.001}, False),
    "no_check": (777, {"neigh_check": False, "neigh_every": 5, "skin": 0.001}, False),
    "close_band": (1111, {"skin": 0.00004, "cdf": 1.1}, False),
    "gravity_last": (1025, {"gravity_first": 0}, False),
    "sibling": (1500, SIBLING, False),
    "epsd2": (1500, EPSD2, False),
    "mesh": (1025, {}, True),
    "mesh_gravity_last": (1025, dict(EPSD2, gravity_first=0), True),
    "four_lanes": (17_001, {"skin": 0.001}, False),
    "four_lanes_long_rows": (16_500, {"skin": 0.0033}, False),
}


def _system(n, change, mesh, precision):
    params, mats, P, walls = wl.dense_pack(seed=n, n=n, rolling=True, speed=0.2, periodic=(0, 0, 0))
    lo, hi = params["boxlo"], params["boxhi"]
    params = dict(params, **change)
    mats = dict(mats, characteristic_velocity=1.0, cohesion_energy_density=[[2e4]])
    walls = walls + [(0, lo[0] + 0.0003, 1), (0, hi[0] - 0.0003, 1), (1, lo[1] + 0.0003, 1), (1, hi[1] - 0.0003, 1)]
    meshes = ()
    if mesh:
        mats = dict(wl.materials_two(rolling_friction=0.1))
        walls = []
        x = P["x"]
        # a margin just under the smallest radius: the outermost spheres overlap
        # the drum, and no centre lies on it (a contact without a normal)
        margin = 0.0009
        radius = 0.5 * float(np.hypot(*(x[:, :2].max(0) - x[:, :2].min(0)))) + margin
        tris = np.asarray(msh.drum(radius, float(x[:, 2].max() - x[:, 2].min()) + 2 * margin, 24, 4))
        c = 0.5 * (x.max(0) + x.min(0))
        P = dict(P, x=x - c)  # the drum is centred on the origin, its axis is y
        P["x"] = np.ascontiguousarray(P["x"][:, [0, 2, 1]])
        b = 4.0 * radius
        params.update(boxlo=(-b, -b, -b), boxhi=(b, b, b))
        meshes = [(tris, 2, None, ((0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 0.5))]
    longest = 128 if params["skin"] > 0.003 else 0  # 0: the default limit of 32 entries a row
    return pydem.GpuSystem(params, mats, P, walls, precision=precision, meshes=meshes, max_neighbors=longest)


@pytest.mark.parametrize("precision", [pydem.DEM_FP64, pydem.DEM_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name", list(CASES))
def test_groups_equal_one_lane_bitwise(name, precision):
    n, change, mesh = CASES[name]
    print(f"[gpu] lane groups {name} n={n} precision={precision}", flush=True)
    got = []
    for persist in (0, 4):
        g = _system(n, change, mesh, precision)
        g.set_step_shape(0, persist)
        g.run(60)
        st, stats = g.state(), g.stats()
        got.append((st, stats, None if mesh else g.wall_history(), g.pairs()))
        g.close()
    (sa, ta, wa, pa), (sb, tb, wb, pb) = got
    for k in ("x", "v", "omega", "f", "torque"):
        assert np.isfinite(sa[k]).all(), k
        assert np.array_equal(sa[k], sb[k]), k
    for k in ("npairs", "ncontacts", "nwall_contacts", "nrebuilds"):
        assert ta[k] == tb[k], k
    if not mesh:
        assert np.array_equal(wa, wb)
    for a, b in zip(pa, pb):
        assert np.array_equal(a, b)
    if n > 700:
        assert ta["ncontacts"] > 100
        assert ta["nwall_contacts"] > 0
