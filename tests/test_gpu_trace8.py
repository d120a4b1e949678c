"""The 8-wide traversal at its edges: waves that are partly filled, scenes of one
node or one leaf, steps with more (ray, triangle) pairs than lanes, ties, and
maximum distances at and below 0, at a hit and beyond every hit.  Records must
match the oracle's brute force bit for bit."""
import numpy as np
import pytest

import oracle
from cudapt_amd import scenes
from tests.helpers import hits_equal, random_rays

pytestmark = pytest.mark.gpu


def _triangles(kind):
    rng = np.random.default_rng(5)
    if kind == "one":
        return np.array([[[-1, -1, 0], [1, -1, 0], [0, 1, 0]]], np.float32)
    if kind == "coincident":                        # every ray that meets one meets all: the lowest id wins
        return np.repeat(np.array([[[-2, -2, 0], [2, -2, 0], [0, 3, 0]]], np.float32), 300, 0)
    n = {"nine": 9, "sheets": 500}[kind]
    if kind == "sheets":                            # overlapping sheets: many triangles a step
        z = rng.permutation(n).astype(np.float32)[:, None, None] * 0.004
        t = np.array([[[-2, -2, 0], [2, -2, 0], [0, 3, 0]]], np.float32) + rng.uniform(-0.3, 0.3, (n, 3, 3))
        t[..., 2] = z[..., 0]
        return t.astype(np.float32)
    c = rng.uniform(-1.5, 1.5, (n, 1, 3))
    return (c + rng.uniform(-0.4, 0.4, (n, 3, 3))).astype(np.float32)


@pytest.fixture(scope="module", params=["one", "nine", "coincident", "sheets"])
def scene(request, cpt):
    t = _triangles(request.param)
    sc = scenes.mesh_scene(t.reshape(-1, 3), np.arange(len(t) * 3, dtype=np.uint32).reshape(-1, 3))
    return cpt.Scene(sc), oracle.Scene(sc)


def _hits(cpt, S, rays):
    dr, dh = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(len(rays) * 16)
    S.trace_device(dr.ptr, len(rays), dh.ptr, layout=2)
    return dh.download(oracle.HIT_DTYPE, len(rays))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 5000])
def test_ray_counts(cpt, scene, n):
    S, O = scene
    rays = random_rays(n, [-1, -1, -3], [1, 1, 3], seed=n)
    rays[::2, 4:7] = np.array([0, 0, 1], np.float32) * -np.sign(rays[::2, 2:3])      # straight at the sheets
    ref, _ = O.trace(rays, "brute")
    assert hits_equal(_hits(cpt, S, rays), ref).all()


def test_max_distance(cpt, scene):
    S, O = scene
    rays = random_rays(4096, [-1, -1, -3], [1, 1, 3], seed=3)
    rays[::2, 4:7] = np.array([0, 0, 1], np.float32) * -np.sign(rays[::2, 2:3])
    free, _ = O.trace(rays, "brute")
    hit = free["tri"] != 0xFFFFFFFF
    assert hit.any()
    t = np.where(hit, free["t"], 1.0).astype(np.float32)
    rays[:, 3] = np.choose(np.arange(len(rays)) % 5, [np.float32(0), np.float32(-1), t, np.nextafter(t, np.float32(9)),
                                                     np.float32(1e20)])
    ref, _ = O.trace(rays, "brute")
    assert hits_equal(_hits(cpt, S, rays), ref).all()


@pytest.mark.parametrize("n", [1, 32768, 32769, 500000])
def test_host_queries(cpt, n):
    """Both sides of the pinned staging's bound, and more rays than the persistent grid's lanes."""
    sc = scenes.cornell()
    S, O = cpt.Scene(sc), oracle.Scene(sc)
    rays = random_rays(n, [-0.99, 0.01, -0.99], [0.99, 1.99, 0.99], seed=n)
    ref, _ = O.trace(rays, "brute")
    assert hits_equal(S.trace(rays), ref).all()
