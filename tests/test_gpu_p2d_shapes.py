"""2D problems by size: on both sides of the lines between one, two and four
targets per lane, sorted (far tiles) and shuffled (general loop), a coincident
pair among them, on some of the targets against the FP64 oracle: relative L2 <=
1e-5, the bar of the parity tests."""
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


@pytest.mark.parametrize("shuffled", (False, True))
@pytest.mark.parametrize("reg", ("singular", "planetary", "winckelmans", "gaussian"))
@pytest.mark.parametrize("n", (3001, 16001, 17001, 21001, 41001, 131501))
def test_sizes(orc, n, reg, shuffled):
    case(f"P2D sizes n={n} {reg} shuffled={shuffled}")
    rng = np.random.default_rng(n)
    p, sigma, nu = W.sheet(n)
    sigma, nu = float(np.float32(sigma)), float(np.float32(nu))
    p["vorticity"] *= rng.uniform(0.5, 1.5, n).astype(np.float32)
    p["area"] *= rng.uniform(0.5, 1.5, n).astype(np.float32)
    p["coord"][n // 2] = p["coord"][n // 2 + 700]
    if shuffled:
        p = p[rng.permutation(n)]
    some = np.sort(rng.choice(n, 200, replace=False)).astype(np.int32)
    some[0], some[-1] = 0, n - 1
    visc = reg in ("winckelmans", "gaussian")
    rv, re = orc.f64_P2D(p, p, reg, sigma, nu=nu, idx=some, vel=True, visc=visc)
    v = np.asarray(cv.P2D_M2M_vel(p, p["coord"], reg, sigma), np.float64)
    assert oracle.rel_l2(v[some], rv) <= 1e-5
    if visc:
        e = np.asarray(cv.P2D_M2M_visc_dvort(p, p, reg, sigma, nu), np.float64)
        assert oracle.rel_l2(e[some], re) <= 1e-5
