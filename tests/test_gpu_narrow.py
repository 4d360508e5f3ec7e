"""Small problems, whose waves share 64 targets per workgroup: counts at the
edges of the groups, of a wave's quarter of a tile, of a tile and of the
partitions, and on both sides of the limit, against the FP64 oracle: relative L2
<= 1e-5, the bar of the parity tests, and for the filaments that of the tests
with targets next to a filament (5e-5 or more)."""
import numpy as np
import pytest

import cvortex_amd as cv
import oracle
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu
SIZES = [(1, 1), (63, 64), (64, 65), (65, 63), (193, 129), (257, 255), (513, 1), (1, 700),
         (1023, 257), (4097, 65), (130, 9001),
         (129, 40), (9000, 3), (16500, 70)]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def check(name, got, ref, tol=1e-5):
    got = np.asarray(got, np.float64)
    assert np.all(np.isfinite(got)), name
    assert oracle.rel_l2(got, ref) <= tol, name


@pytest.mark.parametrize("acc", (cv.ACC_COMP, cv.ACC_TILES, cv.ACC_PLAIN))
@pytest.mark.parametrize("ns,nt", SIZES)
def test_edges(orc, ns, nt, acc):
    case(f"narrow ns={ns} nt={nt} acc={acc}")
    p = W.random_p3d(ns, ns, box=1.0, vort=1.0, vol=1.0 / ns)
    t = W.random_p3d(nt, 10000 + nt, box=1.0, vort=1.0, vol=1.0 / nt)
    p2 = W.random_p2d(ns, ns, box=1.0, vort=1.0, area=1.0 / ns)
    t2 = W.random_p2d(nt, 10000 + nt, box=1.0, vort=1.0, area=1.0 / nt)
    f = W.random_f3d(ns, ns, box=1.0, strength=1.0)
    sigma, nu = float(np.float32(0.25)), float(np.float32(1e-3))
    prev = cv.set_accumulation(acc)
    try:
        for reg in ("singular", "winckelmans", "planetary", "gaussian"):
            visc = reg in ("winckelmans", "gaussian")
            got = cv.P3D_M2M_fused(p, t, reg, sigma, nu, visc=visc)
            ref = orc.f64_P3D(p, t, reg, sigma, nu=nu, vel=True, dvort=True, visc=visc)
            for name, g, r in list(zip(("vel", "dvort", "visc"), got, ref))[:3 if visc else 2]:
                check(f"P3D {reg} {name}", g, r)
            r2, e2 = orc.f64_P2D(p2, t2, reg, sigma, nu=nu, vel=True, visc=visc)
            check(f"P2D {reg} vel", cv.P2D_M2M_vel(p2, t2["coord"], reg, sigma), r2)
            if visc:
                check(f"P2D {reg} visc", cv.P2D_M2M_visc_dvort(p2, t2, reg, sigma, nu), e2)
        fv, fd = orc.f64_F3D(f, t)
        # near a filament, 1.5 times the FP32 restatement's own error where that is more
        e = [oracle.rel_l2(a, b) for a, b in ((orc.F3D_M2M_vel(f, t["coord"]), fv),
                                              (orc.F3D_M2M_dvort(f, t), fd))]
        check("F3D vel", cv.F3D_M2M_vel(f, t["coord"]), fv, max(5e-5, 1.5 * e[0]))
        check("F3D dvort", cv.F3D_M2M_dvort(f, t), fd, max(5e-5, 1.5 * e[1]))
    finally:
        cv.set_accumulation(prev)


@pytest.mark.parametrize("n", (8191, 20479, 20481))
def test_limit(orc, n):
    """Both sides of 24 tiles of 256 x 256 per CU on a chip of 256 CUs, and of
    four for the lighter 2D kernels."""
    case(f"narrow limit n={n}")
    p = W.random_p3d(n, n, box=1.0, vort=1.0, vol=1.0 / n)
    p2 = W.random_p2d(n, n, box=1.0, vort=1.0, area=1.0 / n)
    s = float(np.float32(1.5 / n ** (1 / 3)))
    vel, dv = cv.P3D_M2M_fused(p, p, "winckelmans", s)[:2]
    rv, rd = orc.f64_P3D(p, p, "winckelmans", s, vel=True, dvort=True)[:2]
    check("vel", vel, rv)
    check("dvort", dv, rd)
    check("P2D", cv.P2D_M2M_vel(p2, p2["coord"], "planetary", s),
          orc.f64_P2D(p2, p2, "planetary", s, vel=True)[0])
