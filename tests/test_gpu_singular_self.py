"""Singular 3D pairs at one place, which have no value and are left out: in the
targets' own tiles, in others, several in a tile and none, every launch shape and
accumulation, against the FP64 oracle (relative L2 <= 1e-5, the bar of the parity
tests)."""
import numpy as np
import pytest

import cvortex_amd as cv
import oracle
from cvortex_amd import device as D
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("acc", ("ACC_COMP", "ACC_TILES", "ACC_PLAIN"))
@pytest.mark.parametrize("shape", ((1, 1), (2, 3), (4, 2)))
@pytest.mark.parametrize("same", (True, False))
def test_pairs_at_one_place(orc, same, shape, acc):
    case(f"singular pairs at one place same={same} shape={shape} {acc}")
    p = W.random_p3d(1500, 21, box=1.0, vort=1.0)
    for i, j in ((3, 4), (5, 700), (255, 256), (1023, 1499), (10, 1300), (10, 1301)):
        p["coord"][j] = p["coord"][i]
    t = p if same else np.ascontiguousarray(np.concatenate([p[200:900], W.random_p3d(77, 5, box=1.0)]))
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    tv, ta = (pv, a) if same else (D.DeviceArray.from_host(x) for x in D.p3d_soa(t))
    rv, rd = orc.f64_P3D(p, t, "singular", 0.1, gauss_mode=1)[:2]
    for mask in (1, 2, 3):
        out = [D.DeviceArray((len(t), 3)) if mask & b else None for b in (1, 2)]
        D.p3d_eval(D.p3d_problem(pv, a, len(p), tv, ta, len(t), out[0], out[1], None, "singular", 0.1,
                                 accumulate=getattr(cv, acc)), None, shape=shape)
        D.synchronize()
        for o, r in zip(out, (rv, rd)):
            # (close random pairs have strong terms: a plain FP32 sum keeps fewer digits)
            if o:
                assert oracle.rel_l2(o.download(), r) <= (1e-5 if acc != "ACC_PLAIN" else 1e-4)
