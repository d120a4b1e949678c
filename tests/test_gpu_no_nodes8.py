"""A scene with a vertex too far away for the 8-wide nodes' extents is traversed over
the FP32 4-wide nodes: queries match the oracle's brute force bit for bit, layout 2
and Node Format 1 included."""
import numpy as np
import pytest

import oracle
from cudapt_amd import scenes
from tests.helpers import hits_equal, random_rays

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(cpt):
    g = np.random.default_rng(9)
    t = (g.uniform(-2, 2, (300, 1, 3)) + g.uniform(-0.5, 0.5, (300, 3, 3))).astype(np.float32)
    t[0] = [[3e38, 0, 0], [3e38, 1, 0], [3e38, 0, 1]]        # none of its distances is finite: no ray hits it
    with np.errstate(all="ignore"):
        sc = scenes.mesh_scene(t.reshape(-1, 3), np.arange(900, dtype=np.uint32).reshape(-1, 3))
    return cpt.Scene(sc), oracle.Scene(sc)


@pytest.mark.parametrize("cull", [False, True])
@pytest.mark.parametrize("n", [1, 65, 40000])
def test_queries(cpt, scene, n, cull):
    S, O = scene
    rays = random_rays(n, [-2, -2, -2], [2, 2, 2], seed=n)
    rays[::3, 3] = 1.5
    ref, _ = O.trace(rays, "brute", cull=cull)
    assert hits_equal(S.trace(rays, cull=cull), ref).all()
    dr, dh = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(n * 16)
    for layout in (0, 2):
        S.counters(reset=True)
        S.trace_device(dr.ptr, n, dh.ptr, layout=layout, cull=cull)
        assert hits_equal(dh.download(oracle.HIT_DTYPE, n), ref).all()
        cost = S.trace_cost(rays, layout=layout, cull=cull).sum(0, dtype=np.uint64)
        c = S.counters()
        assert (c["nodes"], c["tris"]) == (2 * int(cost[0]), 2 * int(cost[1]))
    S.occluded_device(dr.ptr, n, dh.ptr, cull=cull)
    assert np.array_equal(dh.download(np.uint32, n) != 0, ref["tri"] != 0xFFFFFFFF)
