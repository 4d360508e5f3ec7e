"""Influence matrix of filaments of no length and large strength: 0 for points at their
place and for others, whatever the strength, and no other column changes."""
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


@pytest.mark.parametrize("strength", (1.0, 1e25, 3e38))
@pytest.mark.parametrize("nf,nm", [(3, 40), (700, 130)])
def test_no_length(nf, nm, strength):
    case(f"influence no length nf={nf} nm={nm} strength={strength}")
    rng = np.random.default_rng(nf)
    fl = chains(nf, rng)
    bad = np.unique(np.concatenate([[0], rng.integers(0, nf, nf // 50)]))
    pts = rng.normal(size=(nm, 3)).astype(np.float32)
    dirs = rng.normal(size=(nm, 3)).astype(np.float32)
    want = evaluate(fl, pts, dirs)
    end, g = fl["end"].copy(), fl["strength"].copy()
    end[bad] = fl["start"][bad]
    g[bad] = strength
    keep = np.setdiff1d(np.arange(nf), bad)
    got = evaluate(make_f3d(fl["start"], end, g), pts, dirs)
    assert not np.any(got[:, bad])          # NaN would count as nonzero
    np.testing.assert_allclose(got[:, keep], want[:, keep], rtol=1e-4,
                               atol=1e-5 * np.abs(want[:, keep]).max())
    pts[: len(bad)] = fl["start"][bad][:nm]
    got = evaluate(make_f3d(fl["start"], end, g), pts, dirs)
    assert not np.any(got[:, bad])
