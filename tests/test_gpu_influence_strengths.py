"""Influence matrix of filaments whose strength is not finite: their columns are 0,
for points near them and far away (the element's two forms), for a matrix written
through the caches and one written past them, and no other column changes."""
import numpy as np
import pytest

from cvortex_amd.types import make_f3d
from gpuutil import case, have_gpu
from test_gpu_influence_forms import chains, evaluate

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


@pytest.mark.parametrize("nf,nm", [(3, 40), (700, 130), (8192, 8192)])
def test_non_finite_strengths(nf, nm):
    case(f"influence strengths nf={nf} nm={nm}")
    rng = np.random.default_rng(nf)
    fl = chains(nf, rng)
    k = rng.integers(0, nf, nm)
    off = rng.normal(size=(nm, 3)) * np.exp(rng.uniform(np.log(0.01), np.log(30), (nm, 1)))
    pts = (0.5 * (fl["start"][k] + fl["end"][k]) + off).astype(np.float32)
    dirs = rng.normal(size=(nm, 3)).astype(np.float32)
    want = evaluate(fl, pts, dirs)
    bad = np.unique(np.concatenate([[0], rng.integers(0, nf, 12)]))
    g = fl["strength"].copy()
    g[bad] = np.resize(np.array([np.nan, np.inf, -np.inf], np.float32), len(bad))
    got = evaluate(make_f3d(fl["start"], fl["end"], g), pts, dirs)
    keep = np.setdiff1d(np.arange(nf), bad)
    assert np.array_equal(got[:, keep], want[:, keep])
    assert not np.any(got[:, bad])          # NaN would count as nonzero
