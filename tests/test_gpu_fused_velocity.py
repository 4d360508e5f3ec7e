"""The fused entry points asked for the velocity alone (no strengths of the induced
particles are uploaded), and for the velocity and an exchange that the
regularisation has not, against the FP64 oracle: relative L2 <= 1e-5."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("n", (300, 20000))
def test_velocity_alone(orc, n):
    case(f"fused, velocity alone n={n}")
    p, q = W.random_p3d(n, 1, box=1.0, vort=1.0), W.random_p3d(500, 2, box=1.0, vort=1.0)
    s = float(np.float32(0.1))
    for reg, visc in (("winckelmans", False), ("singular", True)):
        v, d, e = cv.P3D_M2M_fused(p, q, reg, s, 1e-3, vel=True, dvort=False, visc=visc)
        assert d is None and (e is None or not np.any(e))
        assert oracle.rel_l2(v, orc.f64_P3D(p, q, reg, s)[0]) <= 1e-5


def test_filaments(orc):
    case("fused filaments, velocity alone")
    f, q = W.random_f3d(300, 1, box=1.0, strength=1.0), W.random_p3d(500, 2, box=1.0, vort=1.0)
    out = np.zeros((500, 3), np.float32)
    from cvortex_amd.types import pointer_array
    pf, _ = pointer_array(f)
    pq, _ = pointer_array(q)
    assert cv.lib().cvtx_hip_F3D_M2M_fused(pf.ctypes.data, 300, pq.ctypes.data, 500, out.ctypes.data,
                                           None) == 0
    assert np.array_equal(out, cv.F3D_M2M_vel(f, q["coord"]))
