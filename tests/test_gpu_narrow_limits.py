"""The line between 64 and 256 targets per workgroup, 24 tiles of 256 x 256 per CU on
a chip of 256 CUs and 16 for the lighter 2D kernels: 78 x 78 tiles of 256 lie below
the first and 79 x 79 beyond it, 63 x 63 and 64 x 64 at the second.  Against the FP64
oracle, relative L2 <= 1e-5, the bar of the parity tests."""
import numpy as np
import pytest

import cvortex_amd as cv
import oracle
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("n", (78 * 256, 78 * 256 + 1))
def test_3d(orc, n):
    case(f"narrow limit 3D n={n}")
    p = W.random_p3d(n, n, box=1.0, vort=1.0, vol=1.0 / n)
    s = float(np.float32(1.5 / n ** (1 / 3)))
    got = cv.P3D_M2M_fused(p, p, "winckelmans", s)[:2]
    ref = orc.f64_P3D(p, p, "winckelmans", s, vel=True, dvort=True)[:2]
    for g, r in zip(got, ref):
        assert oracle.rel_l2(g, r) <= 1e-5


@pytest.mark.parametrize("n", (63 * 256, 63 * 256 + 1))
@pytest.mark.parametrize("kernel", ("planetary", "singular"))
def test_light_2d(orc, kernel, n):
    case(f"narrow limit 2D {kernel} n={n}")
    p = W.random_p2d(n, n, box=1.0, vort=1.0, area=1.0 / n)
    s = float(np.float32(1.5 / n ** 0.5))
    ref = orc.f64_P2D(p, p, kernel, s, vel=True)[0]
    assert oracle.rel_l2(cv.P2D_M2M_vel(p, p["coord"], kernel, s), ref) <= 1e-5
