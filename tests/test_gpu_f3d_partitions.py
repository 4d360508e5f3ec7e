"""Filament launches around the size from which partitions go down to one tile:
the default shape against one partition.  A partition's sums are added in FP64, so
only the grouping of FP32 tile sums is the same or finer: relative L2 <= 1e-6."""
import numpy as np
import pytest

import cvortex_amd as cv
import oracle
from cvortex_amd import device as D
from cvortex_amd import workloads as W
from cvortex_amd.types import make_f3d
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("nf", (3071, 3072, 3333))
@pytest.mark.parametrize("mask", (1, 2, 3))
def test_default_shape(nf, mask):
    nt = 131073
    case(f"F3D partitions nf={nf} nt={nt} mask={mask}")
    rng = np.random.default_rng(nf)
    a = rng.uniform(0, 1, (nf, 3))
    f = make_f3d(a, a + rng.normal(scale=0.02, size=(nf, 3)), rng.normal(size=nf))
    fa, fb = (D.DeviceArray.from_host(x) for x in D.f3d_soa(f))
    pv, ta = (D.DeviceArray.from_host(x) for x in D.p3d_soa(W.random_p3d(nt, 4, box=1.0, vort=1.0)))
    got = []
    for shape in (None, (1, 1)):
        out = [D.DeviceArray((nt, 3)) if mask & b else None for b in (1, 2)]
        D.f3d_eval(D.F3DProblem(fa.addr, fb.addr, nf, pv.addr, ta.addr, nt,
                                *[o.addr if o else None for o in out], cv.ACC_COMP), None, shape=shape)
        D.synchronize()
        got.append([o.download() for o in out if o])
    for x, y in zip(*got):
        assert oracle.rel_l2(x, y) <= 1e-6
