"""Gaussian 3D pairs at radii for which 1/t^3 or 1/t^2 rounds most (t: the radius times
the power of two that puts it in [1, 2)): the error common to all pairs, the
result's component along the FP64 one less 1, is at most 2^-24.5.  The kernels leave
none of a whole rounding (2^-24 at most, up to 1.5 times that in the exchange): the
table's coefficients round one by one, and the rest of the exponent's factor is kept."""
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


def radii(lo, hi, power):
    """The two radii of 4000 for which t^power rounds most, up and down."""
    s = np.random.default_rng(2).uniform(lo, hi, 4000).astype(np.float32)
    t = s.astype(np.float64) * 2.0 ** -np.floor(np.log2(s))
    v = t ** power * (0.5 / np.log(2) if power == -2 else 1.0)
    d = v.astype(np.float32) / v - 1
    return [float(s[np.argmin(d)]), float(s[np.argmax(d)])]


@pytest.mark.parametrize("shape", (None, (1, 1), (2, 2), (4, 1)))
@pytest.mark.parametrize("sign", (0, 1))
@pytest.mark.parametrize("lo,hi,power", [(2.0, 2.2, -3), (0.55, 0.65, -3), (0.2, 0.25, -2),
                                         (0.3, 0.4, -2)])
def test_common_error(orc, lo, hi, power, sign, shape):
    sigma = radii(lo, hi, power)[sign]
    case(f"gaussian bias sigma={sigma} shape={shape}")
    rng = np.random.default_rng(4)
    n = 2000
    p = make_p3d(rng.uniform(0, 1, (n, 3)), rng.uniform(0.5, 1, (n, 3)), rng.uniform(0.2, 1, n))
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    out = [D.DeviceArray((n, 3)) for _ in range(3)]
    nu = float(np.float32(1e-3))
    D.p3d_eval(D.p3d_problem(pv, a, n, pv, a, n, *out, "gaussian", sigma, nu), None, shape)
    D.synchronize()
    ref = orc.f64_P3D(p, p, "gaussian", sigma, nu, visc=True)
    for name, o, r in zip(("vel", "dvort", "visc"), out, ref):
        if (name == "vel") != (power == -3) or name == "dvort":
            continue
        b = float(np.sum(o.download() * r) / np.sum(r * r) - 1)
        print(f"  {name}: {b:.2e}", flush=True)
        assert abs(b) <= 2.0 ** -24.5, name
