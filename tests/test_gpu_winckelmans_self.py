"""Winckelmans pairs at and near equal coordinates: a tile whose pairs include a
coincident one is summed again with the test, so coincident particles in the
same and in other tiles, distances on both sides of 2^-12 sigma, radii far from
one and every accumulation mode are checked against the FP64 oracle: relative
L2 <= 1e-5, the bar of the parity tests."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd.types import make_p3d
from gpuutil import case, have_gpu
import oracle

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("acc", (cv.ACC_COMP, cv.ACC_TILES, cv.ACC_PLAIN))
@pytest.mark.parametrize("n", (2, 255, 600, 1100))
@pytest.mark.parametrize("scale", (1.0, 3e-7, 2e9))
def test_coincident_and_close(orc, n, scale, acc):
    case(f"winckelmans self n={n} scale={scale} acc={acc}")
    rng = np.random.default_rng(n)
    sigma = 0.3 * scale
    x = rng.uniform(0.1, 1, (n, 3)).astype(np.float32)
    k = n // 4
    x[n - k:] = x[:k]                                     # the same place, often another tile
    m = min(k, 40)
    step = np.exp(rng.uniform(np.log(1e-6), np.log(1e-2), m)) * 0.3
    x[k:k + m] = x[:m] + (step[:, None] * rng.normal(size=(m, 3))).astype(np.float32)
    p = make_p3d((x * np.float32(scale)), rng.normal(size=(n, 3)), rng.uniform(0.5, 1, n) * scale ** 3)
    prev = cv.set_accumulation(acc)
    try:
        got = cv.P3D_M2M_fused(p, p, "winckelmans", sigma, 1e-3, vel=True, dvort=True, visc=True)
    finally:
        cv.set_accumulation(prev)
    ref = orc.f64_P3D(p, p, "winckelmans", float(np.float32(sigma)), float(np.float32(1e-3)),
                      visc=True)
    for name, g, r in zip(("vel", "dvort", "visc"), got, ref):
        assert np.all(np.isfinite(g)), name
        assert oracle.rel_l2(g, r) <= TOL, name
