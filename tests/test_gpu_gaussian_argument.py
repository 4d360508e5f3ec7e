"""Gaussian 3D pairs at radii for which 16/t, the factor of the near range's table
argument, rounds most (t: the radius times the power of two that puts it in [1, 2);
close to 2, where a rounding is 2^-24 of the value).  G falls with up to the third
power of the argument, so a factor taken as it is moves all pairs by up to
3 * 2^-24 the same way; the error common to all, the velocity's component along the
FP64 one less 1, is at most 2^-24.5.  One to four targets per lane; the form with 64
targets per workgroup has no such factor."""
import numpy as np
import pytest

from cvortex_amd import device as D
from cvortex_amd.types import make_p3d
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("shape", ((1, 1), (2, 2), (4, 1)))
@pytest.mark.parametrize("sign", (np.argmin, np.argmax))
@pytest.mark.parametrize("lo,hi", [(0.11, 0.124), (0.225, 0.249)])
def test_common_error(orc, lo, hi, sign, shape):
    s = np.random.default_rng(6).uniform(lo, hi, 4000).astype(np.float32)
    v = 1.0 / s.astype(np.float64)
    sigma = float(s[sign(v.astype(np.float32) / v - 1)])
    case(f"gaussian argument sigma={sigma} shape={shape}")
    rng = np.random.default_rng(4)
    n = 2000
    p = make_p3d(rng.uniform(0, 1, (n, 3)), rng.uniform(0.5, 1, (n, 3)), rng.uniform(0.2, 1, n))
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    out = D.DeviceArray((n, 3))
    D.p3d_eval(D.p3d_problem(pv, a, n, pv, a, n, out, None, None, "gaussian", sigma), None, shape)
    D.synchronize()
    ref = orc.f64_P3D(p, p, "gaussian", sigma, 0.0)[0]
    b = float(np.sum(out.download() * ref) / np.sum(ref * ref) - 1)
    print(f"  common error: {b:.2e}", flush=True)
    assert abs(b) <= 2.0 ** -24.5
