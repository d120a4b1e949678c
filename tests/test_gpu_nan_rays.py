"""Rays with a NaN, or from infinity, hit nothing: they end at the root instead of
visiting every node, and leave the other rays of their wave as they are."""
import numpy as np
import pytest

import oracle
from cudapt_amd import scenes
from tests.helpers import random_rays

pytestmark = pytest.mark.gpu

NAN, INF = np.float32("nan"), np.float32("inf")
# columns of a ray: origin 0-2, direction 4-6, eps 7
BAD = {"direction": ((4, 5, 6), NAN), "direction x": ((4,), NAN), "direction z": ((6,), NAN), "origin": ((0, 1, 2), NAN),
       "origin y": ((1,), NAN), "eps": ((7,), NAN), "far": ((0, 1, 2), INF), "far z": ((2,), -INF)}


@pytest.fixture(scope="module")
def scene(cpt):
    sc = scenes.sphere_grid(grid=16)
    return cpt.Scene(sc)


@pytest.mark.parametrize("kind", list(BAD))
@pytest.mark.parametrize("n,step", [(64, 1), (1000, 1), (5000, 7)])
def test_bad_rays_end_at_the_root(cpt, scene, kind, n, step):
    rays = random_rays(n, [-30, 0.0, -30], [30, 6.0, 30], seed=n)
    dr, dh = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(n * 16)
    scene.trace_device(dr.ptr, n, dh.ptr, layout=2)
    want = dh.download(oracle.HIT_DTYPE, n)
    cost = scene.trace_cost(rays, layout=2)
    bad = np.arange(n) % step == 0
    cols, value = BAD[kind]
    for c in cols:
        rays[bad, c] = value
    dr = cpt.DeviceBuffer.from_array(rays)
    want["tri"][bad], want["t"][bad], want["u"][bad], want["v"][bad] = 0xFFFFFFFF, np.float32(1e20), 0, 0
    cost[bad] = (1, 0)
    for layout in (2, 0):
        scene.counters(reset=True)
        scene.trace_device(dr.ptr, n, dh.ptr, layout=layout)
        c = scene.counters(reset=True)
        got = dh.download(oracle.HIT_DTYPE, n)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        if layout == 2:
            assert c["nodes"] == int(cost[:, 0].sum()) and c["tris"] == int(cost[:, 1].sum())
    assert np.array_equal(scene.trace_cost(rays, layout=2), cost)
    scene.occluded_device(dr.ptr, n, dh.ptr)
    assert not dh.download(np.uint32, n)[bad].any()
