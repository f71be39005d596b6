"""Sizes at which the work splits of three GPU paths can go wrong.

  contact-point solve   eight lanes per pair, eight pairs per wavefront, in
                        batches that give every pair a group of its own: a
                        pair's result does not depend on how many pairs there
                        are (bitwise), and 95 % of the points equal the oracle's
                        to 1e-12 m (the bound of the solve's own test), for
                        integer, half and equal blockiness
  network gradient      16 samples per tile, tiles spread over the wavefronts:
                        1e-3 norm-wise against the checker with the same BF16
                        rounding points (the bound of the network's own test)
  dem_get_state         any subset of the arrays, at block edges
"""
import ctypes

import numpy as np
import pytest

import mlp_oracle as mo
import pydem
import pyoracle as orc
import superquadrics as sq
import workloads as wl

pytestmark = pytest.mark.gpu

SHAPES = {"drawn": None, "ellipsoid": (2.0, 2.0), "integer": (4.0, 6.0), "half": (2.5, 3.5), "equal": (3.0, 3.0)}


@pytest.mark.parametrize("shape", list(SHAPES))
def test_solve_does_not_depend_on_the_batch(shape):
    print(f"[gpu] solve groups, {shape}", flush=True)
    A, B = sq.overlapping_pairs(61, 130)
    if SHAPES[shape]:
        A, B = A.copy(), B.copy()
        A[:, 10:12] = B[:, 10:12] = SHAPES[shape]
    op, *_ = orc.sq_contact_batch(A, B)
    whole = None
    for n in (130, 1, 2, 7, 8, 9, 17, 64, 65):
        s = pydem.SqSolver()
        s.set_pairs(A[:n], B[:n])
        r = s.solve(pydem.DEM_SQ_FRESH)
        again = s.solve(pydem.DEM_SQ_GIVEN, r["point"])
        s.close()
        if whole is None:
            whole = (r, again)
            close = np.linalg.norm(r["point"] - op, axis=1) <= 1e-12
            assert close.mean() >= 0.95
        for full, part in zip(whole, (r, again)):
            for k in ("point", "iters", "flags"):
                assert np.array_equal(full[k][:n], part[k]), (n, k)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 1025])
def test_network_gradient_batch_remainders(n):
    print(f"[gpu] network gradient, batch {n}", flush=True)
    rng = np.random.default_rng(n)
    s = pydem.SqSolver()
    s.net_init(seed=5)
    p = s.net_params()
    p = p + rng.normal(0, 0.05, p.shape).astype(np.float32)
    s.set_net_params(p)
    X = rng.normal(0, 1, (n, 18)).astype(np.float32)
    T = rng.normal(0, 0.5, (n, 3)).astype(np.float32)
    Y = s.net_forward(X)
    g, loss = s.net_gradient(X, T)
    s.close()
    Yc, _ = mo.forward(p, X)
    gc, lc = mo.gradient(p, X, T)
    assert np.linalg.norm(Y - Yc) <= 1e-3 * np.linalg.norm(Yc)
    assert np.linalg.norm(g - gc) <= 1e-3 * np.linalg.norm(gc)
    assert loss == pytest.approx(lc, rel=1e-4)


@pytest.mark.parametrize("precision", [pydem.DEM_FP64, pydem.DEM_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n", [1, 255, 256, 257])
def test_state_subsets(n, precision):
    print(f"[gpu] get_state subsets n={n}", flush=True)
    params, mats, P, walls = wl.dense_pack(seed=n, n=n, periodic=(0, 0, 0))
    g = pydem.GpuSystem(params, mats, P, walls, precision=precision)
    g.run(5)
    names = ("x", "v", "omega", "f", "torque")
    full = g.state()
    dp = ctypes.POINTER(ctypes.c_double)
    for want in range(1, 32):
        out = [np.full((n, 3), -1.0) if (want >> q) & 1 else None for q in range(5)]
        rc = g.lib.dem_get_state(g.h, *[None if o is None else o.ctypes.data_as(dp) for o in out])
        assert rc == 0
        for k, o in zip(names, out):
            assert o is None or np.array_equal(o, full[k]), (want, k)
    g.close()
