"""Filaments of no length in a chain (collapsed panel edges), near the targets and far
from them: the results are those of the chain without them, relative L2 <= 1e-5
against the FP64 oracle, the bar of the far-tile tests."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd import device as D
from cvortex_amd.types import make_f3d, make_p3d
from gpuutil import case, have_gpu
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("gap", (0.3, 40.0))
@pytest.mark.parametrize("shape", (None, (1, 1), (2, 1), (4, 2)))
@pytest.mark.parametrize("mask", (1, 2, 3))
def test_collapsed_edges(orc, mask, shape, gap):
    case(f"F3D no length gap={gap} shape={shape} mask={mask}")
    rng = np.random.default_rng(9)
    n = 300
    pts = np.cumsum(rng.normal(0, 0.1, (n + 1, 3)), axis=0).astype(np.float32)
    flat = np.array([0, 5, 6, 63, 64, 200, 255, 256, 299])
    for i in flat:
        pts[i + 1] = pts[i]
    g = rng.normal(size=n).astype(np.float32)
    g[5] = 0.0
    f = make_f3d(pts[:-1], pts[1:], g)
    x = (rng.uniform(-1, 1, (700, 3)) + pts.mean(axis=0) + [0, 0, gap]).astype(np.float32)
    t = make_p3d(x, rng.normal(size=x.shape), np.ones(len(x)))
    keep = np.linalg.norm(f["end"] - f["start"], axis=1) > 0
    v64, d64 = orc.f64_F3D(np.ascontiguousarray(f[keep]), t)
    fa, fb = (D.DeviceArray.from_host(y) for y in D.f3d_soa(f))
    pv, a = (D.DeviceArray.from_host(y) for y in D.p3d_soa(t))
    v, d = (D.DeviceArray((len(t), 3)) for _ in range(2))
    D.f3d_eval(D.F3DProblem(fa.addr, fb.addr, n, pv.addr, a.addr, len(t), v.addr if mask & 1 else None,
                            d.addr if mask & 2 else None, cv.ACC_COMP), None, shape)
    D.synchronize()
    if mask & 1:
        assert oracle.rel_l2(v.download(), v64) <= 1e-5
    if mask & 2:
        assert oracle.rel_l2(d.download(), d64) <= 1e-5
