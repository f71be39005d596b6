"""After a build that ends in an error the handle keeps the state, the list and
the histories it had. The gap classes of that list must not be trusted any
more: the build has already cleared the distances they are compared with."""
import numpy as np
import pytest

import pydem
import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(0, 0), (0, 4)], ids=["lane_group", "one_lane"])
@pytest.mark.parametrize("precision", [pydem.DEM_FP64, pydem.DEM_MIXED], ids=["fp64", "mixed"])
def test_forces_after_a_lost_atom(precision, shape):
    # a large sphere at rest, a small one that closes a gap of 0.2 mm, and one
    # that leaves the box and asks for a build 0.5 mm (half the skin) later
    r = np.array([0.005, 0.002, 0.001])
    x = np.array([[0.02, 0.02, 0.02], [0.0272, 0.02, 0.02], [0.0397, 0.03, 0.03]])
    v = np.array([[0.0, 0.0, 0.0], [-0.8, 0.0, 0.0], [1.0, 0.0, 0.0]])
    P = {"x": x, "v": v, "omega": np.zeros((3, 3)), "radius": r, "rmass": wl.sphere_mass(r, 2500.0),
         "type": np.ones(3, dtype=np.int32), "tag": np.arange(1, 4, dtype=np.int32)}
    params = {"dt": 5e-6, "skin": 0.001, "cdf": 1.0, "boxlo": (0.0, 0.0, 0.0), "boxhi": (0.04, 0.04, 0.04),
              "periodic": (0, 0, 0), "grav_acc": (0.0, 0.0, 0.0), "gravity_first": 1, "rolling_cdt": 0}
    print(f"[gpu] lost atom, precision {precision}, shape {shape}", flush=True)
    g = pydem.GpuSystem(params, wl.materials_single(), P, [], precision=precision)
    g.set_step_shape(*shape)
    with pytest.raises(Exception, match="Lost atoms"):
        g.run(150)
    g.compute_forces(False)
    s = g.state()
    g.close()
    gap = np.linalg.norm(s["x"][1] - s["x"][0]) - r[0] - r[1]
    assert gap < -1e-5
    assert np.linalg.norm(s["f"][1]) > 0.0
    assert np.allclose(s["f"][0], -s["f"][1], rtol=1e-12, atol=0.0)
