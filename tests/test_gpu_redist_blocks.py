"""Remeshing node sums by blocks of the grid: regions of more particles than one
item holds, cells and blocks at the grid's edges, sparse particles, grids whose
keys are too long for the block bitmaps (the sorted-entry path), strengths that
are not finite, and two calls in a row.  Node sets must be the oracle's bit for
bit.  Strengths are compared with FP64 sums of the same FP32 contributions
(weights in the reference's FP32 operations, formed here in numpy): relative
L2 <= 1e-6, the rounding of the results to FP32 being 6e-8."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd.types import make_p2d, make_p3d
from gpuutil import case, have_gpu
import oracle

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def m4p(U):
    a = F(1) - F(2.5) * U * U + F(1.5) * U * U * U
    b = F(0.5) * (F(1) - U) * (F(2) - U) * (F(2) - U)
    return np.where(U < 1, a, np.where(U < 2, b, F(0)))


def lambda1(U):
    return np.where(U <= 1, F(1) - U, F(0))


def sums(coord, alpha, nodes, h, f):
    """FP64 sums at the nodes of the FP32 contributions of all particles."""
    rh = F(1) / F(h)
    out = np.zeros((len(nodes), alpha.shape[1]))
    for i, x in enumerate(nodes):
        w = [f(np.abs((coord[:, c] - x[c]) * rh)) for c in range(coord.shape[1])]
        frac = w[0] * w[1] if len(w) == 2 else (w[0] * w[1]) * w[2]
        out[i] = (alpha * frac[:, None]).astype(np.float64).sum(0)
    return out


def pick(n, k):
    return np.sort(np.random.default_rng(n).choice(n, min(n, k), replace=False))


@pytest.mark.parametrize("r,f", [("m4p", m4p), ("lambda1", lambda1)])
@pytest.mark.parametrize("n,h,spread", [(1, 0.1, 1.0), (64, 0.05, 1.0), (3000, 0.3, 1.0),
                                        (20001, 0.4, 1.0), (5000, 0.02, 1.0), (300, 0.004, 3.0),
                                        (300, 0.0005, 1.0)])
def test_p3d_blocks(orc, r, f, n, h, spread):
    # 20001 particles on 0.4: about 27 blocks with up to 20001 particles in
    # reach (ten items); 0.0005: 2000 nodes per axis, 33-bit keys
    case(f"P3D blocks {r} n={n} h={h}")
    rng = np.random.default_rng(n)
    p = make_p3d(rng.uniform(0, spread, (n, 3)), rng.normal(size=(n, 3)), np.full(n, 1e-3))
    got = cv.P3D_redistribute_on_grid(p, r, h)
    ref = orc.P3D_redistribute_on_grid(p, r, h)
    assert len(got) == len(ref) and np.array_equal(got["coord"], ref["coord"])
    assert np.array_equal(got["volume"], ref["volume"])
    k = pick(len(got), 300)
    assert oracle.rel_l2(got["vorticity"][k],
                         sums(p["coord"], p["vorticity"], got["coord"][k], h, f)) <= 1e-6
    again = cv.P3D_redistribute_on_grid(p, r, h)
    assert np.array_equal(again, got)


@pytest.mark.parametrize("n,h", [(1, 0.1), (70, 0.05), (30011, 0.2), (4000, 0.004), (200, 2e-5)])
def test_p2d_blocks(orc, n, h):
    # 2e-5: 50000 nodes per axis, 32-bit keys
    case(f"P2D blocks n={n} h={h}")
    rng = np.random.default_rng(n)
    q = make_p2d(rng.uniform(0, 1, (n, 2)), rng.normal(size=n), np.full(n, 1e-3))
    got = cv.P2D_redistribute_on_grid(q, "m4p", h)
    ref = orc.P2D_redistribute_on_grid(q, "m4p", h)
    assert len(got) == len(ref) and np.array_equal(got["coord"], ref["coord"])
    k = pick(len(got), 300)
    a = q["vorticity"].reshape(-1, 1)
    assert oracle.rel_l2(got["vorticity"][k].reshape(-1, 1),
                         sums(q["coord"], a, got["coord"][k], h, m4p)) <= 1e-6
    assert np.array_equal(cv.P2D_redistribute_on_grid(q, "m4p", h), got)


@pytest.mark.parametrize("value", (np.nan, np.inf))
@pytest.mark.parametrize("negligible", (0.0, 0.1))
def test_strength_that_is_not_finite(value, negligible):
    # the mean strength and the removal threshold are then not finite either,
    # and no node is stronger: nothing is left
    case(f"P3D blocks with a strength of {value}, negligible={negligible}")
    rng = np.random.default_rng(8)
    p = make_p3d(rng.uniform(0, 1, (2000, 3)), rng.normal(size=(2000, 3)), np.full(2000, 1e-3))
    p["vorticity"][77, 1] = value
    assert len(cv.P3D_redistribute_on_grid(p, "m4p", 0.05, negligible=negligible)) == 0
