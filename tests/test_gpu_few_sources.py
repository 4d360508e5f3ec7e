"""Few sources on many targets and few targets of many sources, on both sides of the
lines between the launch forms: sampled targets against the FP64 oracle, relative
L2 <= 1e-5, the bar of the parity tests (5e-5 for filaments, which pass close)."""
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


@pytest.mark.parametrize("ns,nt", [(1, 262145), (63, 32769), (64, 32769), (300, 261889), (700, 300001),
                                   (300001, 1), (262144, 65), (150000, 600), (140000, 2049)])
def test_counts(orc, ns, nt):
    case(f"{ns} sources on {nt} targets")
    p = W.random_p3d(ns, 1, box=1.0, vort=1.0, vol=1.0 / ns)
    t = W.random_p3d(nt, 2, box=1.0, vort=1.0, vol=1.0 / nt)
    p2 = W.random_p2d(ns, 1, box=1.0, vort=1.0, area=1.0 / ns)
    t2 = W.random_p2d(nt, 2, box=1.0, vort=1.0, area=1.0 / nt)
    idx = np.unique(np.concatenate([[0, nt - 1], np.random.default_rng(3).integers(0, nt, 40)]))
    idx = idx.astype(np.int32)
    sub = lambda x: np.ascontiguousarray(x[idx])
    sigma, nu = float(np.float32(0.1)), float(np.float32(1e-3))
    for reg in ("winckelmans", "gaussian"):
        got = cv.P3D_M2M_fused(p, t, reg, sigma, nu, visc=True)
        ref = orc.f64_P3D(p, sub(t), reg, sigma, nu=nu, visc=True)
        for name, g, r in zip(("vel", "dvort", "visc"), got, ref):
            assert oracle.rel_l2(g[idx], r) <= 1e-5, (reg, name)
    for reg in ("planetary", "gaussian", "winckelmans"):
        v = cv.P2D_M2M_vel(p2, t2["coord"], reg, sigma)
        assert oracle.rel_l2(v[idx], orc.f64_P2D(p2, sub(t2), reg, sigma, vel=True)[0]) <= 1e-5, reg
    e = cv.P2D_M2M_visc_dvort(p2, t2, "gaussian", sigma, nu)
    r = orc.f64_P2D(p2, sub(t2), "gaussian", sigma, nu=nu, vel=True, visc=True)[1]
    assert oracle.rel_l2(e[idx], r) <= 1e-5
    w = cv.P3D_M2M_vort(p, t["coord"], "gaussian", sigma)
    assert oracle.rel_l2(w[idx], orc.f64_P3D_vort(p, sub(t)["coord"], "gaussian", sigma)) <= 1e-5
    if ns <= 1000 or nt <= 100:
        f = W.random_f3d(min(ns, 20000), 1, box=1.0, strength=1.0)
        fv = orc.f64_F3D(f, sub(t))[0]
        assert oracle.rel_l2(cv.F3D_M2M_vel(f, t["coord"])[idx], fv) <= 5e-5
