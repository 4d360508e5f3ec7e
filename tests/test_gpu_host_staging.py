"""Calls on host arrays at the edges of how their data moves (outputs written
straight to pinned memory up to 64 KB, copies by a kernel up to 1 MiB, by HIP
beyond): the same bits as the device-resident entry point gives for the same
particles, and unchanged by a larger and a smaller call in between."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd import device as D
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def resident(p, t, dvort):
    spv, sa = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    tpv, ta = (D.DeviceArray.from_host(x) for x in D.p3d_soa(t))
    v = D.DeviceArray((len(t), 3))
    d = D.DeviceArray((len(t), 3)) if dvort else None
    D.p3d_eval(D.p3d_problem(spv, sa, len(p), tpv, ta, len(t), v, d, None, "winckelmans", 0.1))
    D.synchronize()
    return [x.download() for x in (v, d) if x]


# 5461 x 12 bytes is the last output below 64 KB; 2 x 30037 + 5462 (or 2 x 5462)
# float4 are the first inputs above 1 MiB
@pytest.mark.parametrize("nt", (1, 3, 2730, 2731, 5461, 5462))
@pytest.mark.parametrize("ns", (1, 5, 700, 30037))
def test_host_call_equals_resident(ns, nt):
    case(f"host staging ns={ns} nt={nt}")
    p, t = W.random_p3d(ns, 5, box=1.0, vort=1.0), W.random_p3d(nt, 6, box=1.0, vort=1.0)
    seam = cv.lib().cvtx_hip_set_dispatch(1)  # the device for every size
    try:
        for rep in range(2):
            v, d, _ = cv.P3D_M2M_fused(p, t, "winckelmans", 0.1, 0.0, vel=True, dvort=True)
            rv, rd = resident(p, t, True)
            assert np.array_equal(v, rv) and np.array_equal(d, rd)
            assert np.array_equal(cv.P3D_M2M_vel(p, t["coord"], "winckelmans", 0.1),
                                  resident(p, t, False)[0])
            other = W.random_p3d(4000 if rep == 0 else 9, 7, box=1.0, vort=1.0)
            cv.P3D_M2M_vel(other, other["coord"], "gaussian", 0.1)
    finally:
        cv.lib().cvtx_hip_set_dispatch(seam)
