"""dem_get_state takes no device memory: a system that fills the card can be
read out. It reorders the arrays in the state buffer that the next step writes
whole, so reading the state between steps changes nothing in them."""
import numpy as np
import pytest
import torch

import pydem
import workloads as wl

pytestmark = pytest.mark.gpu
PRECISIONS = {"fp64": pydem.DEM_FP64, "mixed": pydem.DEM_MIXED}


@pytest.mark.parametrize("precision", list(PRECISIONS))
def test_reading_the_state_takes_no_device_memory(precision):
    params, mats, P, walls = wl.settling_1m(seed=2, n=400_000)
    g = pydem.GpuSystem(params, mats, P, walls, precision=PRECISIONS[precision])
    g.run(2)
    print(f"[gpu] state of 400,000 spheres, {precision}", flush=True)
    before = torch.cuda.mem_get_info()[0]
    g.state()
    after = torch.cuda.mem_get_info()[0]
    g.close()
    # all five arrays are 48 MB
    assert before - after < 4 << 20


@pytest.mark.parametrize("precision", list(PRECISIONS))
def test_reading_the_state_changes_no_step(precision):
    params, mats, P, walls = wl.dense_pack(seed=4, n=3001, periodic=(0, 0, 0))
    out = []
    for read in (False, True):
        print(f"[gpu] runs of odd and even length, state read between: {read}", flush=True)
        g = pydem.GpuSystem(params, mats, P, walls, precision=PRECISIONS[precision])
        for steps in (7, 8, 1, 40):
            g.run_continue(steps) if steps != 7 else g.run(steps)
            if read:
                g.state()
        out.append(g.state())
        g.close()
    for k in ("x", "v", "omega", "f", "torque"):
        assert np.array_equal(out[0][k], out[1][k]), k
