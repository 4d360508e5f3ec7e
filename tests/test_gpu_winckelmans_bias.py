"""Winckelmans pairs at radii whose square rounds most: the error common to all pairs,
which no averaging removes (the result's component along the FP64 one, less 1).
With d <= 2^-24 the rounding of sigma^2, the kernels are built to leave
  exchange, uniform neighbourhood: 0 on average; all pairs in the core: 1.5 d
  velocity: 0.6 d and the rounding of 1.5 sigma^2, 0.6 of 2^-24
and the constants' and sums' rounding adds at most 2^-25, so 2^-23 and 2^-23.3 bound
them (rounding sigma^2 alone gives up to 4.5 d and 1.5 d)."""
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


def radii(lo, hi):
    """The two radii of 4000 whose squares round most, up and down."""
    s = np.random.default_rng(1).uniform(lo, hi, 4000).astype(np.float32)
    s2 = s.astype(np.float64) ** 2
    d = s2.astype(np.float32) / s2 - 1
    return [float(s[np.argmin(d)]), float(s[np.argmax(d)])]


@pytest.mark.parametrize("shape", (None, (1, 1), (2, 2)))
@pytest.mark.parametrize("sign", (0, 1))
@pytest.mark.parametrize("lo,hi", [(0.2, 0.3), (0.5, 0.6), (2.0, 2.2)])
def test_common_error(orc, lo, hi, sign, shape):
    sigma = radii(lo, hi)[sign]
    case(f"winckelmans bias sigma={sigma} shape={shape}")
    rng = np.random.default_rng(4)
    n = 2000
    p = make_p3d(rng.uniform(0, 1, (n, 3)), rng.uniform(0.5, 1, (n, 3)), rng.uniform(0.2, 1, n))
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    out = [D.DeviceArray((n, 3)) for _ in range(3)]
    nu = float(np.float32(1e-3))
    D.p3d_eval(D.p3d_problem(pv, a, n, pv, a, n, *out, "winckelmans", sigma, nu), None, shape)
    D.synchronize()
    ref = orc.f64_P3D(p, p, "winckelmans", sigma, nu, visc=True)
    for name, o, r, bound in zip(("vel", "dvort", "visc"), out, ref, (2 ** -23.3, None, 2.0 ** -23)):
        b = float(np.sum(o.download() * r) / np.sum(r * r) - 1)
        print(f"  {name}: {b:.2e}", flush=True)
        assert bound is None or abs(b) <= bound, name
