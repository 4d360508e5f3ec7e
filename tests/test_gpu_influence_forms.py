"""The influence-matrix kernel's two element forms and its stores: points
from a tenth of a filament's length to far away in one call (so that waves
take the far form for some rows and the general form for others), points on
filament lines and end points, non-finite points, odd and even column counts,
partial column blocks, and a matrix large enough to be written past the
caches.  Tolerance: relative L2 <= 1e-5 against the FP64 oracle, the bar of
the other influence tests."""
import numpy as np
import pytest

from cvortex_amd import device as D
from cvortex_amd.types import make_f3d
from gpuutil import case, have_gpu
import oracle

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def evaluate(fl, pts, dirs):
    def soa(x):
        y = np.zeros((len(x), 4), np.float32)
        y[:, :3] = x
        return D.DeviceArray.from_host(y)
    fa, fb = (D.DeviceArray.from_host(x) for x in D.f3d_soa(fl))
    out = D.DeviceArray((len(pts), len(fl)))
    D.f3d_inf_eval(fa, fb, len(fl), soa(pts), soa(dirs), len(pts), out)
    return out.download()


def chains(n, rng, ny=32):
    """Filaments in polylines of ny segments, 0.02-0.05 long."""
    a = np.zeros((n, 3), np.float32)
    b = np.zeros((n, 3), np.float32)
    for c in range(0, n, ny):
        m = min(ny, n - c)
        steps = np.concatenate([rng.uniform(-1, 1, (1, 3)), rng.normal(0, 0.02, (m, 3))])
        line = np.cumsum(steps, axis=0).astype(np.float32)
        a[c:c + m], b[c:c + m] = line[:-1], line[1:]
    return make_f3d(a, b, rng.normal(size=n).astype(np.float32))


@pytest.mark.parametrize("nf,nm", [(1, 33), (511, 65), (512, 64), (514, 31), (923, 130), (2048, 700)])
def test_near_and_far_rows(orc, nf, nm):
    case(f"influence forms nf={nf} nm={nm}")
    rng = np.random.default_rng(nf + nm)
    fl = chains(nf, rng)
    k = rng.integers(0, nf, nm)
    length = np.linalg.norm(fl["end"][k] - fl["start"][k], axis=1, keepdims=True)
    off = rng.normal(size=(nm, 3))
    off *= length * np.exp(rng.uniform(np.log(0.1), np.log(1e3), (nm, 1))) / np.linalg.norm(
        off, axis=1, keepdims=True)
    pts = (0.5 * (fl["start"][k] + fl["end"][k]) + off).astype(np.float32)
    pts[0] = fl["end"][k[0]]                                     # an end point
    pts[1] = 2.0 * fl["end"][k[1]] - fl["start"][k[1]]           # on a line's extension
    dirs = rng.normal(size=(nm, 3)).astype(np.float32)
    got = evaluate(fl, pts, dirs)
    ref = orc.f64_F3D_inf_mtrx(fl, pts, dirs)
    # columns of the filaments that rows 0 and 1 lie on: FP32 coordinates
    # decide which side of "exactly on the line" a point is
    for r in (0, 1):
        got[r], ref[r] = 0.0, 0.0
    assert np.all(np.isfinite(got))
    assert oracle.rel_l2(got, ref) <= TOL


def test_non_finite_rows_stay_their_own():
    # a NaN or infinite point makes its own row NaN and no other
    case("influence with non-finite points")
    rng = np.random.default_rng(5)
    fl = chains(700, rng)
    pts = rng.uniform(-1, 1, (40, 3)).astype(np.float32)
    dirs = rng.normal(size=(40, 3)).astype(np.float32)
    want = evaluate(fl, pts, dirs)
    bad = pts.copy()
    bad[7, 1], bad[20, 0] = np.nan, np.inf
    got = evaluate(fl, bad, dirs)
    assert np.all(np.isnan(got[[7, 20]]))
    keep = [i for i in range(40) if i not in (7, 20)]
    assert np.array_equal(got[keep], want[keep])


def test_streamed_matrix(orc):
    # 8192 x 8192 floats: 256 MiB, rows of whole 128-byte lines
    case("influence 8192 x 8192")
    rng = np.random.default_rng(6)
    fl = chains(8192, rng)
    pts = rng.uniform(-1, 1, (8192, 3)).astype(np.float32)
    dirs = rng.normal(size=(8192, 3)).astype(np.float32)
    got = evaluate(fl, pts, dirs)
    rows = np.sort(rng.choice(8192, 24, replace=False)).astype(np.int32)
    assert oracle.rel_l2(got[rows], orc.f64_F3D_inf_mtrx(fl, pts, dirs, idx=rows)) <= TOL
    assert np.all(np.isfinite(got))
