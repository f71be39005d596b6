"""Large packed beds are walked by the XCDs in stretches of 64 tiles instead of
16 (dem_system.cpp, step_stretch). Which workgroup steps a particle does not
change a bit of it: the rule's shape is compared with grids whose tiles are
divided otherwise -- another tile size, and a persistent grid that holds less
than one round of stretches -- just below and above the size where the rule
changes, with a remainder after the whole rounds, and from captured graphs."""
import numpy as np
import pytest

import pydem
import workloads as wl

pytestmark = pytest.mark.gpu

MANY = 256 * 1024


def _run(system, shape, graphs, steps):
    params, mats, P, walls = system
    g = pydem.GpuSystem(params, mats, P, walls, precision=pydem.DEM_MIXED)
    g.set_step_shape(*shape)
    g.set_graph_capture(graphs)
    g.run(steps)
    out, stats = g.state(), g.stats()
    g.close()
    return out, stats


@pytest.mark.parametrize("n", [MANY - 1, MANY, 300_001])
def test_stretches_change_no_bit(n):
    system = wl.packed_1m(seed=n, n=n)
    print(f"[gpu] packed bed of {n}: default shape", flush=True)
    ref, rstats = _run(system, (0, 0), False, 70)
    assert rstats["npairs"] >= 3 * n and rstats["ncontacts"] > n
    for shape, graphs in (((3, 0), False), ((0, 1), False), ((0, 0), True)):
        print(f"[gpu] shape {shape} graphs {graphs}", flush=True)
        got, gstats = _run(system, shape, graphs, 70)
        for k in ("x", "v", "omega", "f", "torque"):
            assert np.array_equal(ref[k], got[k]), (shape, k)
        for k in ("npairs", "ncontacts", "nwall_contacts", "nrebuilds"):
            assert rstats[k] == gstats[k], (shape, k)
