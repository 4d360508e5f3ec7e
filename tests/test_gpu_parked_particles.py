"""Particles parked at the largest float: as sources they contribute nothing, as
targets they get nothing, at every radius (Gaussian positions are multiplied by a
power of two), launch shape and in batches."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd import device as D
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu
FAR = np.finfo(np.float32).max


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def evaluate(s, t, reg, sigma, shape, acc):
    spv, sa = (D.DeviceArray.from_host(x) for x in D.p3d_soa(s))
    tpv, ta = (D.DeviceArray.from_host(x) for x in D.p3d_soa(t))
    out = [D.DeviceArray((len(t), 3)) for _ in range(3)]
    D.p3d_eval(D.p3d_problem(spv, sa, len(s), tpv, ta, len(t), *out, reg, sigma, 1e-3, acc), None,
               shape)
    D.synchronize()
    return [o.download() for o in out]


@pytest.mark.parametrize("acc", (cv.ACC_COMP, cv.ACC_TILES, cv.ACC_PLAIN))
@pytest.mark.parametrize("shape", (None, (1, 1), (2, 1), (4, 2)))
@pytest.mark.parametrize("sigma", (0.02, 1e-5, 3.0))
@pytest.mark.parametrize("reg", ("gaussian",))
def test_parked(reg, sigma, shape, acc):
    case(f"parked particles {reg} sigma={sigma} shape={shape} acc={acc}")
    s, t = W.random_p3d(600, 5, box=1.0, vort=0.1), W.random_p3d(300, 6, box=1.0, vort=0.1)
    still = s.copy()
    still["vorticity"][590:] = 0          # the same tiles without the parked ones' strengths
    still["volume"][590:] = 0
    s["coord"][590:] = FAR
    t["coord"][[7, 250]] = FAR
    got = evaluate(s, t, reg, sigma, shape, acc)
    want = evaluate(still, t, reg, sigma, shape, acc)
    near = np.ones(len(t), bool)
    near[[7, 250]] = False
    for name, g, w in zip(("vel", "dvort", "visc"), got, want):
        assert np.array_equal(g[near], w[near]), name
        assert not np.any(g[~near]), name


@pytest.mark.parametrize("reg", ("gaussian",))
def test_batch(reg):
    case(f"parked particles in a batch {reg}")
    p = W.random_p3d(300, 8, box=1.0, vort=0.1)
    p["coord"][200:210] = FAR
    b = D.Batch(np.array([0, 300], np.int32), np.array([0.02], np.float32), reg)
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    out = [D.DeviceArray((300, 3)) for _ in range(2)]
    b.eval(pv, a, *out)
    D.synchronize()
    for o in out:
        x = o.download()
        assert np.all(np.isfinite(x)) and not np.any(x[200:210])
    b.destroy()
