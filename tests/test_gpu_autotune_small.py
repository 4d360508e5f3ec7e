"""The autotuner on problems small enough for 64 targets per workgroup: what it
returns is one of the shapes that two numbers name, and evaluating that shape and
the recorded one agree with the FP64 oracle (relative L2 <= 1e-5)."""
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


@pytest.mark.parametrize("n", (700, 1000, 3000))
def test_returned_shape(orc, n):
    case(f"autotuner n={n}")
    L = cv.lib()
    p = W.random_p3d(n, n, box=1.0, vort=1.0)
    dev = D.P3DDevice(p)
    outs = dev.outputs(True, True, False)
    prob = dev.problem(outs, "winckelmans", 0.3)
    ref = orc.f64_P3D(p, p, "winckelmans", float(np.float32(0.3)))
    tiles = -(-n // 256)
    L.cvtx_hip_tune_clear()
    try:
        T, k, ms = D.autotune_p3d(prob, 20)
        print(f"  {T} targets per lane, {k} partitions, {ms:.4f} ms", flush=True)
        # (as launched: partitions of whole tiles, none empty)
        assert T in (1, 2, 4) and ms > 0
        assert k in {-(-tiles // -(-tiles // q)) for q in range(1, tiles + 1)}
        for shape in ((T, k), None):
            D.p3d_eval(prob, None, shape)
            D.synchronize()
            for o, r in zip(outs[:2], ref):
                assert oracle.rel_l2(o.download(), r) <= 1e-5
    finally:
        L.cvtx_hip_tune_clear()
