"""Radii that are no length, Winckelmans and Gaussian, in every launch shape and in
batches: 0 and NaN give NaN, an infinite one gives 0."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd import device as D
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def expected(x, sigma):
    return np.all(x == 0) if np.isinf(sigma) else np.all(np.isnan(x))


@pytest.mark.parametrize("sigma", (np.nan, 0.0, np.inf))
@pytest.mark.parametrize("shape", (None, (1, 1), (2, 1), (4, 2)))
@pytest.mark.parametrize("acc", (cv.ACC_COMP, cv.ACC_TILES))
@pytest.mark.parametrize("reg", ("winckelmans", "gaussian"))
def test_no_length(reg, acc, shape, sigma):
    case(f"radius {sigma} {reg} shape={shape} acc={acc}")
    s, t = W.random_p3d(600, 1, box=1.0, vort=1.0), W.random_p3d(300, 2, box=1.0, vort=1.0)
    spv, sa = (D.DeviceArray.from_host(x) for x in D.p3d_soa(s))
    tpv, ta = (D.DeviceArray.from_host(x) for x in D.p3d_soa(t))
    for mask in (1, 2, 7):
        out = [D.DeviceArray((len(t), 3)) if mask >> i & 1 else None for i in range(3)]
        D.p3d_eval(D.p3d_problem(spv, sa, len(s), tpv, ta, len(t), *out, reg, sigma, 1e-3, acc),
                   None, shape)
        D.synchronize()
        for name, o in zip(("vel", "dvort", "visc"), out):
            if o is not None:
                assert expected(o.download(), sigma), (name, mask)


@pytest.mark.parametrize("shape", (None, (1, 4), (2, 4)))
@pytest.mark.parametrize("reg", ("winckelmans", "gaussian"))
def test_batch(reg, shape):
    case(f"radii of a batch {reg} shape={shape}")
    p = W.random_p3d(300, 3, box=1.0, vort=1.0)
    sig = np.array([np.nan, 0.0, np.inf], np.float32)
    b = D.Batch(np.array([0, 100, 200, 300], np.int32), sig, reg)
    if shape:
        b.set_shape(*shape)
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    out = [D.DeviceArray((300, 3)) for _ in range(2)]
    b.eval(pv, a, *out)
    D.synchronize()
    for o in out:
        x = o.download()
        for c in range(3):
            assert expected(x[100 * c:100 * c + 100], sig[c]), (c, reg)
    b.destroy()
