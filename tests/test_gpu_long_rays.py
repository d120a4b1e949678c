"""Maximum distances past 1e20, the distance IntersectTri gives a missed triangle:
the answer is then that "hit" of the lowest triangle tested, as the reference's
arithmetic has it.  The rays meet the boxes of all triangles, so the oracle's brute
force tests the same ones."""
import numpy as np
import pytest

import oracle
from cudapt_amd import scenes
from tests.helpers import hits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("maxd", [1e20, 2e20, np.inf])
@pytest.mark.parametrize("n", [1, 100, 40000])
def test_missed_triangles(cpt, maxd, n):
    t = np.array([[[-1, -1, 0], [1, -1, 0], [1, 1, 0]], [[-1, -1, 0], [1, 1, 1], [1, -1, 0]]], np.float32)
    sc = scenes.mesh_scene(t.reshape(-1, 3), np.arange(6, dtype=np.uint32).reshape(-1, 3))
    S, O = cpt.Scene(sc), oracle.Scene(sc)
    rng = np.random.default_rng(n)
    rays = np.zeros((n, 8), np.float32)
    rays[:, :2], rays[:, 2], rays[:, 3] = rng.uniform(-0.99, 0.99, (n, 2)), 5, maxd
    rays[:, 4:8] = 0, 0, -1, 1e-4
    ref, _ = O.trace(rays, "brute")
    assert hits_equal(S.trace(rays), ref).all()
    dr, dh = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(n * 16)
    S.trace_device(dr.ptr, n, dh.ptr, layout=0)
    assert hits_equal(dh.download(oracle.HIT_DTYPE, n), ref).all()
    S.occluded_device(dr.ptr, n, dh.ptr)
    assert np.array_equal(dh.download(np.uint32, n) != 0, ref["tri"] != 0xFFFFFFFF)


@pytest.mark.parametrize("maxd", [1e20, 3e38])
def test_missed_triangles_of_layout_2(cpt, maxd):
    t = np.array([[[-1, -1, 0], [1, -1, 0], [1, 1, 0]]], np.float32)
    sc = scenes.mesh_scene(t.reshape(-1, 3), np.arange(3, dtype=np.uint32).reshape(-1, 3))
    S, O = cpt.Scene(sc), oracle.Scene(sc)
    rays = np.zeros((500, 8), np.float32)
    rays[:, :2], rays[:, 2], rays[:, 3] = np.random.default_rng(0).uniform(-0.99, 0.99, (500, 2)), 5, maxd
    rays[:, 4:8] = 0, 0, -1, 1e-4
    ref, _ = O.trace(rays, "brute")
    dr, dh = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(500 * 16)
    S.trace_device(dr.ptr, 500, dh.ptr, layout=2)
    assert hits_equal(dh.download(oracle.HIT_DTYPE, 500), ref).all()
