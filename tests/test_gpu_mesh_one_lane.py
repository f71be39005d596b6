"""Meshes in the step of large systems: one lane a particle, which stops after
the plane walls and leaves the particles with candidate triangles to a packed
launch of their own (k_step_mesh). Systems as small as the tests' would take
the lane groups, which do the meshes in place; a persistent grid (shape 0, 4)
keeps one lane. The mesh tests against the oracle are run again in that shape,
and what they leave out is compared with the lane groups: plane walls beside a
mesh, the counts per instance, the mesh totals, captured graphs, the movers."""
import numpy as np
import pytest

import meshes as msh
import pydem
import test_gpu_batched
import test_gpu_models
import test_gpu_parity
import test_gpu_wall_local
import workloads as wl

pytestmark = pytest.mark.gpu

P, M, B, W = test_gpu_parity, test_gpu_models, test_gpu_batched, test_gpu_wall_local
AGAINST_ORACLE = {
    **{f"floor_one_step_{m}": (P.test_mesh_floor_one_step_fp64, (m,))
       for m in (False, True, "linear", "wiggle", "viblin", "vibrot")},
    "floor_many_steps": (P.test_mesh_floor_many_steps_fp64, ()),
    "floor_close_band": (P.test_mesh_floor_contact_distance_factor_fp64, ()),
    **{f"moving_floor_{m}": (P.test_translating_floor_many_steps_fp64, (m,))
       for m in ("linear", "wiggle", "viblin", "vibrot")},
    "drum_fp64": (P.test_rotating_drum, (pydem.DEM_FP64,)),
    "drum_mixed": (P.test_rotating_drum, (pydem.DEM_MIXED,)),
    "drum_in_pieces": (P.test_rotating_drum_run_in_pieces, ()),
    **{f"graphs_{c}": (P.test_graph_capture_is_bitwise_eager, (c,)) for c in ("drum", "wiggle", "vibrot")},
    "stress": (P.test_mesh_stress_totals_match_oracle, ()),
    "own_model": (M.test_mesh_wall_with_its_own_model_fp64, ()),
    "epsd2_fp64": (M.test_mesh_wall_epsd2, (pydem.DEM_FP64,)),
    "epsd2_mixed": (M.test_mesh_wall_epsd2, (pydem.DEM_MIXED,)),
    "instances_alone": (B.test_batched_instances_equal_alone_bitwise, ()),
    "instance_oracle": (B.test_batched_instance_matches_oracle_fp64, ()),
    "wall_local": (W.test_wall_local_matches_oracle, (True, pydem.DEM_FP64)),
}


@pytest.mark.parametrize("name", list(AGAINST_ORACLE))
def test_against_oracle(name, monkeypatch):
    made = pydem.GpuSystem.__init__

    def init(self, *args, **kw):
        made(self, *args, **kw)
        self.set_step_shape(0, 4)

    monkeypatch.setattr(pydem.GpuSystem, "__init__", init)
    print(f"[gpu] one lane a particle: {name}", flush=True)
    test, args = AGAINST_ORACLE[name]
    test(*args)


MOVERS = {"still": None, "rotate": ((0.0, 0.0, 0.0), (0.0, 0.0, 1.0), 0.05),
          "wiggle": {"wiggle": ((0.00003, 0.0, 0.00005), 0.01)}}


@pytest.mark.parametrize("change", [{}, {"cdf": 1.15}, {"gravity_first": 0}], ids=["plain", "close_band", "gravity_last"])
@pytest.mark.parametrize("mover", list(MOVERS))
@pytest.mark.parametrize("precision", [pydem.DEM_FP64, pydem.DEM_MIXED], ids=["fp64", "mixed"])
def test_walls_and_instances_beside_a_mesh(precision, mover, change):
    # three instances of one box: a tessellated floor below four plane walls
    params, _, Q, _ = wl.dense_pack(seed=12, n=1700, rolling=True, periodic=(0, 0, 0), speed=0.3)
    lo, hi = params["boxlo"], params["boxhi"]
    walls = [(0, lo[0] + 0.0003, 2), (0, hi[0] - 0.0003, 2), (1, lo[1] + 0.0003, 2), (1, hi[1] - 0.0003, 2)]
    floor = msh.grid(lo[0] - 0.002, hi[0] + 0.002, lo[1] - 0.002, hi[1] + 0.002, lo[2], 7, 6)
    meshes = [(floor, 2, {"rolling_cdt": 1}, MOVERS[mover], (0.0, 0.0, 0.0))]
    params = dict(params, skin=0.0001, **change)
    mats = [wl.materials_two(rolling_friction=0.1), wl.materials_two(mu_pw=0.2, rolling_friction=0.1),
            wl.materials_two(restitution=0.6, rolling_friction=0.1)]
    got = []
    for shape, graphs in (((0, 0), False), ((0, 4), False), ((0, 4), True)):
        print(f"[gpu] walls and mesh, {mover}, shape {shape}, graphs {graphs}", flush=True)
        g = pydem.GpuSystem(params, mats[0], Q, walls, precision=precision, meshes=meshes,
                            instances=[700, 1, 999], instance_materials=mats)
        g.set_step_shape(*shape)
        g.set_graph_capture(graphs)
        g.run(111)
        g.run_continue(90)
        got.append((g.state(), g.stats(), g.wall_history(), g.mesh_history(), g.instance_stats(), g.mesh_force(),
                    g.mesh_nodes()))
        g.close()
    ref = got[0]
    assert ref[1]["nwall_contacts"] > 100 and (ref[3][0] >= 0).sum() > 20 and np.abs(ref[2]).max() > 0
    for one in got[1:]:
        for k in ("x", "v", "omega", "f", "torque"):
            assert np.array_equal(ref[0][k], one[0][k]), k
        for k in ("npairs", "ncontacts", "nwall_contacts", "nrebuilds"):
            assert ref[1][k] == one[1][k], k
        assert np.array_equal(ref[2], one[2])
        for part in (3, 4, 6):
            for a, b in zip(ref[part], one[part]):
                assert np.array_equal(a, b), part
        for a, b in zip(ref[5], one[5]):  # FP64 atomics: the order of the additions differs
            assert np.linalg.norm(a - b) <= 1e-11 * np.linalg.norm(a)
