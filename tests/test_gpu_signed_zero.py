"""Pairs at one place whose coordinates differ in the sign of a zero (-0.0 against
+0.0, as for image particles at a symmetry plane) are coincident: no stretching and
no exchange between them.  Winckelmans and Gaussian, sources and targets each way,
every launch shape and accumulation, and batches, against the FP64 oracle: relative
L2 <= 1e-5, the bar of the parity tests."""
import numpy as np
import pytest

import cvortex_amd as cv
import oracle
from cvortex_amd import device as D
from cvortex_amd.types import make_p3d
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu
SIGMA, NU = float(np.float32(0.3)), float(np.float32(1e-3))


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def images(n, negative):
    """Particles on a coordinate plane each, and as many at the same places with the
    other zero; `negative`: the sign of the first ones' zeros."""
    rng = np.random.default_rng(n)
    x = rng.uniform(0.1, 1, (n, 3)).astype(np.float32)
    y = x.copy()
    plane = (np.arange(n), rng.integers(0, 3, n))
    x[plane], y[plane] = (-0.0, 0.0) if negative else (0.0, -0.0)
    def mk(c):
        return make_p3d(c, rng.normal(size=(n, 3)), rng.uniform(0.5, 1, n))
    return mk(x), mk(y)


@pytest.mark.parametrize("acc", (cv.ACC_COMP, cv.ACC_TILES, cv.ACC_PLAIN))
@pytest.mark.parametrize("shape", (None, (1, 1), (2, 1), (4, 2)))
@pytest.mark.parametrize("negative", (False, True))
@pytest.mark.parametrize("reg", ("winckelmans", "gaussian"))
def test_opposite_zeros(orc, reg, negative, shape, acc):
    case(f"signed zero {reg} negative sources={negative} shape={shape} acc={acc}")
    s, t = images(600, negative)
    ref = orc.f64_P3D(s, t, reg, SIGMA, NU, visc=True)
    spv, sa = (D.DeviceArray.from_host(x) for x in D.p3d_soa(s))
    tpv, ta = (D.DeviceArray.from_host(x) for x in D.p3d_soa(t))
    for mask in (7, 2, 1):
        out = [D.DeviceArray((len(t), 3)) if mask >> i & 1 else None for i in range(3)]
        D.p3d_eval(D.p3d_problem(spv, sa, len(s), tpv, ta, len(t), *out, reg, SIGMA, NU, acc),
                   None, shape)
        D.synchronize()
        for name, o, r in zip(("vel", "dvort", "visc"), out, ref):
            if o is not None:
                assert oracle.rel_l2(o.download(), r) <= 1e-5, (name, mask)


@pytest.mark.parametrize("shape", (None, (1, 4), (2, 4)))
@pytest.mark.parametrize("reg", ("winckelmans", "gaussian"))
def test_batch(orc, reg, shape):
    case(f"signed zero in a batch {reg} shape={shape}")
    p = np.concatenate(images(300, False))
    n = len(p)
    b = D.Batch(np.array([0, n], np.int32), np.array([SIGMA], np.float32), reg, outputs=7, nu=NU)
    if shape:
        b.set_shape(*shape)
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    out = [D.DeviceArray((n, 3)) for _ in range(3)]
    b.eval(pv, a, *out)
    D.synchronize()
    for name, o, r in zip(("vel", "dvort", "visc"), out, orc.f64_P3D(p, p, reg, SIGMA, NU, visc=True)):
        assert oracle.rel_l2(o.download(), r) <= 1e-5, name
    b.destroy()
