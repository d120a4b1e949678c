"""The cross-bilateral filter at its edges: images of partial tiles, the largest
radius whose halo lies in LDS and the smallest beyond, guides so sharp that
whole waves of taps weigh 0, infinite and NaN inputs, and the depth term with
and without the albedo guide.  Bit for bit against the oracle's defined arithmetic."""
import numpy as np
import pytest

import oracle
from cudapt_amd import scenes

pytestmark = pytest.mark.gpu


def _same(a, b):
    a, b = a.view(np.uint32), b.view(np.uint32)
    nan = np.isnan(a.view(np.float32)) & np.isnan(b.view(np.float32))
    return bool((nan | (a == b)).all())


@pytest.mark.parametrize("radius,W,H", [(1, 1, 1), (2, 17, 16), (8, 33, 15), (9, 48, 31), (10, 31, 33), (5, 130, 70)])
@pytest.mark.parametrize("diff", [False, True])
@pytest.mark.parametrize("odd", [False, True])
def test_tiles(cpt, radius, W, H, diff, odd):
    rng = np.random.default_rng(radius)
    col = rng.uniform(0, 2, (H, W, 3)).astype(np.float32)
    nrm = rng.normal(size=(H, W, 3)).astype(np.float32)
    dif = rng.uniform(0, 1, (H, W, 3)).astype(np.float32)
    # positions in plateaus: exponents of 0 within one, far past 103 across
    pos = np.repeat(((np.arange(W)[None, :] // 40 + np.arange(H)[:, None] // 20) * 50.0)[..., None], 3, -1).astype(np.float32)
    if odd:
        for a in (col, pos, nrm):
            a[rng.integers(H), rng.integers(W), 1] = np.inf
            a[rng.integers(H), rng.integers(W), 2] = np.nan
    N = rng.integers(1, 60, (H, W)).astype(np.uint32)
    sig = (0.5, 0.4, 0.25, 0.1)
    d = dif if diff else None
    f, _ = cpt.filter_cross_bilateral(col, pos, nrm, d, N, *sig, radius, nd=5)
    assert _same(f, oracle.bilateral_defined(col, pos, nrm, d, *sig, radius))


@pytest.mark.parametrize("radius", [3, 9, 11])
@pytest.mark.parametrize("diff", [0, 1])
def test_depth(cpt, radius, diff):
    sc = scenes.cornell()
    S = cpt.Scene(sc)
    W, H = 61, 43
    R = cpt.Renderer(W, H, mode=cpt.CPT_MODE_BDPT_ADAPTIVE_PLL, **{
        "Filter Radius": radius, "Filter Diffuse Flag": diff, "Filter Depth EuD": 0.05, "Filter Spatial EuD": 2.5,
        "Filter Color EuD": 0.3, "Filter Pos EuD": 0.5})
    col = R.render(S, sc["camera"], frames=5)       # the warm-up: the image the next frame's filter reads
    g = [R.read(b) for b in (cpt.CPT_BUF_GBUF_POS, cpt.CPT_BUF_GBUF_NORM, cpt.CPT_BUF_GBUF_DIFF)]
    R.render(S, sc["camera"], frames=1)
    got = R.read(cpt.CPT_BUF_FILTERED)
    ref = oracle.bilateral_ext(col, g[0], g[1], g[2] if diff else None, 0.3, 0.5, 0.25, 0.1, radius, ss=2.5, sz=0.05,
                               cam=sc["camera"]["pos"])
    assert _same(got, ref)


@pytest.mark.parametrize("radius,diff,depth", [(3, 0, 0.05), (9, 0, 0.05), (7, 0, 0.0), (4, 1, 0.05), (10, 0, 0.05)])
def test_pair(cpt, radius, diff, depth):
    """The learned modes filter the second moment in the image's pass; a profiled renderer filters it on its own."""
    sc = scenes.cornell()
    S = cpt.Scene(sc)
    M = cpt.Mlp(3)
    got = []
    for prof in (True, False):
        R = cpt.Renderer(67, 45, mode=cpt.CPT_MODE_BDPT_ADAPTIVE_PLL, **{
            "Filter Radius": radius, "Filter Diffuse Flag": diff, "Filter Depth EuD": depth, "Filter Color EuD": 0.3,
            "Filter Pos EuD": 0.5, "Learned Signal": 3})
        R.set_profiling(prof)
        R.set_mlp(M)
        img = R.render(S, sc["camera"], frames=8)
        got.append([img] + [R.read(b) for b in (cpt.CPT_BUF_FILTERED, cpt.CPT_BUF_ERROR, cpt.CPT_BUF_ALLOC_ERROR,
                                                cpt.CPT_BUF_SAMPLE_COUNTS)])
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
