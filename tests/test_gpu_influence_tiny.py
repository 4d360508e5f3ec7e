"""Influence matrix at distances whose squares are denormal or zero in FP32: points
that close to a filament's end, and filaments of that length, give finite elements,
and an ordinary filament's column is right (relative L2 <= 1e-5 against the FP64
oracle, the bar of the influence tests).  The points nearly lie on the line of one
filament, whose elements the oracle itself forms by cancellation (8.9e-3 for one of
about 1e-15): that column is only asked to be finite."""
import numpy as np
import pytest

from cvortex_amd.types import make_f3d
from gpuutil import case, have_gpu
from test_gpu_influence_forms import evaluate
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("linked", (False, True))
@pytest.mark.parametrize("length", (1.0, 1e-12, 1e-17, 1e-20, 1e-23, 0.0))
def test_tiny_distances(orc, length, linked):
    case(f"influence tiny length={length} linked={linked}")
    rng = np.random.default_rng(3)
    d = np.concatenate([10.0 ** np.arange(-45.0, -8.0), [0.0, 0.1, 3.0]])
    u = rng.normal(size=(len(d), 3))
    pts = (d[:, None] * u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
    e = np.array([1.0, 0.0, 0.0]) * length
    a = np.array([[0, 0, 0], e if linked else [0, 0, 0], [1, 1, 1], [2, 2, 2]], np.float32)
    b = np.array([e, 2 * e if linked else -e, [2, 2, 2], [1, 3, 1]], np.float32)
    fl = make_f3d(a, b, np.ones(4, np.float32))
    dirs = rng.normal(size=pts.shape).astype(np.float32)
    got = evaluate(fl, pts, dirs)
    assert np.all(np.isfinite(got))
    assert oracle.rel_l2(got[:, 3], orc.f64_F3D_inf_mtrx(fl, pts, dirs)[:, 3]) <= 1e-5
