"""The sorted vorticity-field kernel's queues and partitions: source counts that
leave a partial chunk or queue block, partitions with few or no chunks, every
targets-per-lane value, radii for which no, some and all pairs are within the
cut-off, and coordinates that are not finite.  Tolerance: relative L2 <= 1e-6
against the unsorted kernel, which sums the same pairs in another order (the
bar of the sorted-against-unsorted test), and <= 1e-5 against the oracle on
sampled targets: the FP64 one, since the restatement's FP32 sum over tens of
thousands of one-signed terms is itself 2.6e-5 off, except for the planetary
core, whose edge is defined by the restatement's FP32 arithmetic."""
import numpy as np
import pytest

import cvortex_amd as cv
from cvortex_amd import device as D
from cvortex_amd import workloads as W
from cvortex_amd.types import REG_ID
from gpuutil import case, have_gpu
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def field(p, x, k, sigma, shape=None, order=1, acc=cv.ACC_COMP):
    pv, a = (D.DeviceArray.from_host(y) for y in D.p3d_soa(p))
    t = np.zeros((len(x), 4), np.float32)
    t[:, :3] = x
    dt, out = D.DeviceArray.from_host(t), D.DeviceArray((len(x), 3))
    prev = cv.lib().cvtx_hip_set_target_order(order)
    try:
        D.vort_eval(D.VortProblem(pv.addr, a.addr, len(p), dt.addr, len(x), out.addr, REG_ID[k],
                                  sigma, acc), shape=shape)
        D.synchronize()
    finally:
        cv.lib().cvtx_hip_set_target_order(prev)
    return out.download()


@pytest.mark.parametrize("k", ("winckelmans", "planetary", "gaussian"))
@pytest.mark.parametrize("ns,nt,sigma,shape", [
    (65537, 1025, 0.01, None), (20003, 5000, 0.003, (1, 1)), (20003, 5000, 0.02, (2, 7)),
    (20003, 5000, 0.02, (4, 1)), (66000, 1100, 0.1, (1, 256)), (20003, 5000, 0.3, None)])
def test_sorted_matches_unsorted(orc, k, ns, nt, sigma, shape):
    case(f"vort sorted {k} ns={ns} nt={nt} sigma={sigma} shape={shape}")
    p = W.random_p3d(ns, 900 + ns, box=1.0, vort=1.0)
    x = W.random_p3d(nt, 901 + nt, box=1.1, vort=1.0)["coord"]
    got = field(p, x, k, sigma, shape)
    brute = field(p, x, k, sigma, order=0)
    assert np.all(np.isfinite(got))
    assert oracle.rel_l2(got, brute) <= 1e-6
    idx = np.random.default_rng(3).choice(nt, 64, replace=False)
    ref = (orc.P3D_M2M_vort(p, x[idx], k, sigma) if k == "planetary"
           else orc.f64_P3D_vort(p, x[idx], k, sigma))
    assert oracle.rel_l2(got[idx], ref) <= 1e-5


def test_sorted_plain_accumulation():
    case("vort sorted, one FP32 sum")
    p = W.random_p3d(20003, 911, box=1.0, vort=1.0)
    x = W.random_p3d(5000, 912, box=1.0, vort=1.0)["coord"]
    got = field(p, x, "gaussian", 0.02, acc=cv.ACC_PLAIN)
    assert oracle.rel_l2(got, field(p, x, "gaussian", 0.02)) <= 1e-6


def test_sorted_non_finite_coordinates():
    # a source that is nowhere contributes nothing, a target that is nowhere
    # gets nothing, and neither disturbs the others
    case("vort sorted with non-finite coordinates")
    p = W.random_p3d(20003, 921, box=1.0, vort=1.0)
    x = W.random_p3d(5000, 922, box=1.0, vort=1.0)["coord"]
    bad = [5, 700, 19999, 20002]
    q = p.copy()
    q["coord"][bad[0], 0], q["coord"][bad[1], 1] = np.nan, np.inf
    q["coord"][bad[2]], q["coord"][bad[3], 2] = np.nan, -np.inf
    y = x.copy()
    y[7], y[4000, 2], y[4999, 0] = np.nan, np.inf, np.nan
    gone = p.copy()
    gone["vorticity"][bad] = 0
    got, want = field(q, y, "gaussian", 0.03), field(gone, x, "gaussian", 0.03)
    assert np.all(got[[7, 4000, 4999]] == 0)
    keep = np.setdiff1d(np.arange(5000), [7, 4000, 4999])
    assert np.all(np.isfinite(got))
    assert oracle.rel_l2(got[keep], want[keep]) <= 1e-6
