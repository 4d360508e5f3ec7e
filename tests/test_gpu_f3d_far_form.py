"""The filament kernels' far-tile form at its limits: target blocks just beyond
half the longest filament from a tile (where S^2 - L^2 cancels most), chains
that break at the edges of the link words (64 filaments) and tiles (256),
filament counts that leave a partial group, and every targets-per-lane value.
Tolerance: relative L2 <= 1e-5 against the FP64 oracle (the far-tile bar)."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd import device as D
from cvortex_amd.types import make_f3d, make_p3d
from gpuutil import case, have_gpu
import oracle

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def run(f, t, mask, T):
    fa, fb = (D.DeviceArray.from_host(x) for x in D.f3d_soa(f))
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(t))
    v = D.DeviceArray((len(t), 3)) if mask & cv.OUT_VEL else None
    d = D.DeviceArray((len(t), 3)) if mask & cv.OUT_DVORT else None
    D.f3d_eval(D.F3DProblem(fa.addr, fb.addr, len(f), pv.addr, a.addr, len(t),
                            v.addr if v else None, d.addr if d else None, cv.ACC_COMP),
               None, shape=(T, 1))
    return (v.download() if v else None), (d.download() if d else None)


@pytest.mark.parametrize("mask", (1, 2, 3))
@pytest.mark.parametrize("T", (1, 2, 4))
@pytest.mark.parametrize("nf,gap", [(1, 0.55), (65, 0.55), (257, 0.6), (300, 30.0)])
def test_far_form_limits(orc, nf, gap, T, mask):
    case(f"F3D far form nf={nf} gap={gap} T={T} mask={mask}")
    rng = np.random.default_rng(nf)
    # a chain of unit segments in the box [0, 2]^3, broken at word and tile edges
    p = np.zeros((nf + 1, 3))
    for i in range(nf):
        for _ in range(100):
            step = rng.normal(size=3)
            q = p[i] + step / np.linalg.norm(step)
            if np.all((q >= 0) & (q <= 2)):
                break
        p[i + 1] = np.clip(q, 0, 2)
    a, b = p[:-1].astype(np.float32), p[1:].astype(np.float32)
    for i in (31, 62, 63, 64, 127, 255, 256):
        if i < nf:
            b[i] = rng.uniform(0, 2, 3)
    f = make_f3d(a, b, rng.normal(size=nf).astype(np.float32))
    longest = np.linalg.norm(f["end"] - f["start"], axis=1).max()
    x = rng.uniform(0, 2, (256 * T + 3, 3)).astype(np.float32)
    x[:, 2] = 2.0 + gap * longest + rng.uniform(0, 0.1, len(x))
    t = make_p3d(x, rng.normal(size=x.shape), np.ones(len(x)))
    v, d = run(f, t, mask, T)
    v64, d64 = orc.f64_F3D(f, t)
    if mask & 1:
        assert oracle.rel_l2(v, v64) <= TOL
    if mask & 2:
        assert oracle.rel_l2(d, d64) <= TOL
