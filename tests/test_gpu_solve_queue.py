"""Groups of the contact-point solve that take a second pair. A launch has at
most 2,048 wavefronts of eight groups, so above 16,384 pairs a group starts a
new pair with what the last one left in its registers and LDS columns, while
the other groups of its wavefront are in the middle of theirs. A pair's result
is the same bits in a batch of 20,000, in slices that give every pair a group
of its own, and wherever it stands in the batch."""
import numpy as np
import pytest

import pydem
import superquadrics as sq

pytestmark = pytest.mark.gpu

N, SLICE = 20_000, 8_000


@pytest.fixture(scope="module")
def pairs():
    return sq.overlapping_pairs(79, N)


def _solve(A, B, start, init=None):
    s = pydem.SqSolver()
    s.set_pairs(A, B)
    r = s.solve(start, init)
    s.close()
    return r


@pytest.mark.parametrize("start", ["fresh", "given"])
def test_solve(pairs, start):
    A, B = pairs
    kind = pydem.DEM_SQ_FRESH if start == "fresh" else pydem.DEM_SQ_GIVEN
    # given points somewhere near the pair: some of these solves fall back to the homotopy
    rng = np.random.default_rng(2)
    init = None if start == "fresh" else 0.5 * (A[:, :3] + B[:, :3]) + rng.normal(0, 3e-4, (N, 3))
    take = lambda ix: None if init is None else init[ix]  # noqa: E731
    print(f"[gpu] {N} pairs {start}", flush=True)
    whole = _solve(A, B, kind, init)
    if start == "given":
        assert 0 < ((whole["flags"] >> 1) & 1).sum() < N
    order = rng.permutation(N)
    moved = _solve(A[order], B[order], kind, take(order))
    parts = [_solve(A[k:k + SLICE], B[k:k + SLICE], kind, take(slice(k, k + SLICE))) for k in range(0, N, SLICE)]
    for k in ("point", "fi", "fj", "iters", "flags"):
        assert np.array_equal(whole[k][order], moved[k]), k
        assert np.array_equal(whole[k], np.concatenate([p[k] for p in parts])), k


def test_check(pairs):
    """Contact detection, every third pair with its boxes apart: those are
    passed over by the groups that fetch the next pair. The second call starts
    from the first one's history."""
    A, B = pairs
    B = B.copy()
    B[::3, :3] *= 4.0
    rng = np.random.default_rng(3)
    vel, mass = rng.normal(0, 0.1, (N, 12)), rng.uniform(1e-5, 2e-5, (N, 2))

    def run(ix):
        s = pydem.SqSolver()
        s.set_pairs(A[ix], B[ix])
        first = s.check()
        hist = first["hist"].copy()
        second = s.check(hist, vel[ix], mass[ix], 1e-5)
        s.close()
        return first, second

    print(f"[gpu] check of {N} pairs", flush=True)
    whole = run(np.arange(N))
    apart = (whole[0]["flags"] >> 2) & 1
    assert apart[::3].mean() > 0.9 and apart.sum() < N // 2
    order = rng.permutation(N)
    moved = run(order)
    parts = [run(np.arange(k, min(k + SLICE, N))) for k in range(0, N, SLICE)]
    for c in range(2):
        for k in ("hist", "contact", "en", "deltan", "cp_i", "cp_j", "point", "fi", "fj", "iters", "flags"):
            assert np.array_equal(whole[c][k][order], moved[c][k]), (c, k)
            assert np.array_equal(whole[c][k], np.concatenate([p[c][k] for p in parts])), (c, k)
