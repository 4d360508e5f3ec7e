"""Batches with 64 targets per workgroup (the default of small batches) and with
one target per lane: clouds at the edges of groups, blocks and tiles, empty ones
among them, particles at the same place in one tile and in two, every output and
accumulation, against the FP64 oracle (relative L2 <= 1e-5, the bar of the parity
tests); and the shape cache's column for the variant."""
import numpy as np
import pytest

import cvortex_amd as cv
import oracle
from cvortex_amd import device as D
from cvortex_amd import workloads as W
from gpuutil import case, have_gpu

pytestmark = pytest.mark.gpu
SIZES = (0, 1, 2, 63, 64, 65, 0, 255, 256, 257, 511, 513, 700)


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not have_gpu():
        pytest.fail("no HIP device: GPU tests need one")


def clouds():
    off = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.int32)
    p = W.random_p3d(int(off[-1]), 17, box=1.0, vort=1.0, vol=1e-3)
    for b, n in zip(off, SIZES):
        if n >= 65:
            p["coord"][b + 60] = p["coord"][b + 3]         # one tile
            p["coord"][b + n - 1] = p["coord"][b + 1]      # the first and the last tile
    return p, off, np.linspace(0.05, 0.9, len(SIZES)).astype(np.float32)


@pytest.mark.parametrize("shape", (None, (1, 4), (2, 4)))
@pytest.mark.parametrize("outputs", (3, 7))
@pytest.mark.parametrize("acc", ("ACC_COMP", "ACC_TILES", "ACC_PLAIN"))
@pytest.mark.parametrize("kernel", ("winckelmans", "gaussian"))
def test_cloud_sizes(orc, kernel, acc, outputs, shape):
    case(f"batch of small clouds {kernel} {acc} outputs={outputs} shape={shape}")
    p, off, sig = clouds()
    n = len(p)
    pv, a = (D.DeviceArray.from_host(x) for x in D.p3d_soa(p))
    b = D.Batch(off, sig, kernel, outputs=outputs, nu=0.01, accumulate=getattr(cv, acc))
    if shape:
        b.set_shape(*shape)
    else:
        assert b.shape()[:2] == (1, 256)
    out = [D.DeviceArray((n, 3)) for _ in range(3 if outputs & 4 else 2)]
    b.eval(pv, a, *out)
    D.synchronize()
    got = [o.download() for o in out]
    for c, m in enumerate(SIZES):
        if m == 0:
            continue
        cl = np.ascontiguousarray(p[off[c]:off[c + 1]])
        ref = orc.f64_P3D(cl, cl, kernel, float(sig[c]), 0.01, gauss_mode=1, visc=True)
        for g, r in zip(got, ref):
            g = g[off[c]:off[c + 1]]
            if not np.any(r):
                assert not np.any(g)
            else:
                assert oracle.rel_l2(g, r) <= 1e-5, (m, kernel, acc)
    b.destroy()


def test_cached_variant(tmp_path):
    # a line with the column 4 gives that variant back, one with a shape it does
    # not go with the ordinary one
    case("shape cache: 64 targets per workgroup")
    p, off, sig = clouds()
    sizes = np.diff(off).astype(np.int64)
    key = f"3 1 3 1 {int((sizes * sizes).sum()).bit_length() - 1} {len(sig).bit_length() - 1}"
    L = cv.lib()
    try:
        for line, units in (("1 8 0.0 256 4", 64), ("1 8 0.0 256", 256), ("2 8 0.0 256 4", 512)):
            path = tmp_path / "shapes.txt"
            path.write_text(f"{key} {line}\n")
            L.cvtx_hip_tune_clear()
            assert L.cvtx_hip_tune_load(str(path).encode()) == 1
            b = D.Batch(off, sig, "winckelmans")
            assert b.info()[0] == sum(-(-m // units) for m in SIZES)
            assert L.cvtx_hip_tune_save(str(path).encode()) == 0
            assert (len(path.read_text().split()) == 11) == (units == 64)
            b.destroy()
    finally:
        L.cvtx_hip_tune_clear()
