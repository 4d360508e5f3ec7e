"""A cached shape of 64 targets per workgroup, met by the smallest counts of its
bucket: no targets (nothing to do), no sources (zeros), one of each."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd import device as D
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("ns,nt", [(2000, 0), (2000, 1), (0, 1), (0, 0), (1, 1)])
def test_counts(orc, tmp_path, ns, nt):
    case(f"cached four-wave shape with {ns} sources, {nt} targets")
    s, t = W.random_p3d(max(ns, 1), 1, box=1.0, vort=1.0), W.random_p3d(max(nt, 1), 2, box=1.0, vort=1.0)
    path = tmp_path / "shapes.txt"
    path.write_text(f"0 1 1 1 {max(ns, 1).bit_length() - 1} 0 1 4 0.0 256 4\n")
    L = cv.lib()
    spv, sa = (D.DeviceArray.from_host(x) for x in D.p3d_soa(s))
    tpv, ta = (D.DeviceArray.from_host(x) for x in D.p3d_soa(t))
    out = D.DeviceArray.from_host(np.full((1, 3), 7.0, np.float32))
    try:
        L.cvtx_hip_tune_clear()
        assert L.cvtx_hip_tune_load(str(path).encode()) == 1
        D.p3d_eval(D.p3d_problem(spv, sa, ns, tpv, ta, nt, out, None, None, "winckelmans", 0.3))
        D.synchronize()
    finally:
        L.cvtx_hip_tune_clear()
    got = out.download()
    if nt == 0:
        assert np.all(got == 7.0)
    elif ns == 0:
        assert not np.any(got)
    else:
        ref = orc.f64_P3D(s, t, "winckelmans", float(np.float32(0.3)))[0]
        assert oracle.rel_l2(got, ref) <= 1e-5
