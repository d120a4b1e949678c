"""Rays that touch a triangle's edge within rounding, where the FP32 4-wide
nodes' box test culls the triangle and the conservative 8-wide one does not.
Queries without a layout, and layout 0, answer as the FP32 nodes do; layout 2
gives the minimum of (t, id) over all triangles.  The rays, and the FP32 nodes'
answers, were recorded from a kernel that traversed those nodes alone."""
import os

import numpy as np
import pytest

import oracle
from cudapt_amd import scenes
from tests.helpers import hits_equal

pytestmark = pytest.mark.gpu

GOLDEN = np.load(os.path.join(os.path.dirname(__file__), "golden", "edge_rays.npz"))


@pytest.fixture(scope="module", params=["grid", "cornell"])
def scene(request, cpt):
    sc = scenes.sphere_grid() if request.param == "grid" else scenes.cornell()
    return request.param, cpt.Scene(sc), oracle.Scene(sc)


@pytest.mark.parametrize("cull", [False, True])
@pytest.mark.parametrize("repeat", [1, 40000])       # every lane's ray traced again, and past one chunk a wave
def test_closest(cpt, scene, cull, repeat):
    name, S, O = scene
    at = GOLDEN[name + "_closest_cull"] == cull
    rays = np.tile(GOLDEN[name + "_closest_rays"][at], (repeat, 1))
    want = np.tile(GOLDEN[name + "_closest_ans"][at], (repeat, 1))
    assert np.array_equal(S.trace(rays, cull=cull).view(np.uint32).reshape(-1, 4), want)
    dr, dh = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(len(rays) * 16)
    S.trace_device(dr.ptr, len(rays), dh.ptr, layout=0, cull=cull)
    assert np.array_equal(dh.download(np.uint32, len(rays) * 4).reshape(-1, 4), want)
    S.trace_device(dr.ptr, len(rays), dh.ptr, layout=2, cull=cull)
    n = int(at.sum())
    ref, _ = O.trace(rays[:n], "brute", cull=cull)
    got = dh.download(oracle.HIT_DTYPE, len(rays)).reshape(repeat, n)
    assert all(hits_equal(g, ref).all() for g in got[:: max(1, repeat // 50)])


@pytest.mark.parametrize("cull", [False, True])
def test_occluded(cpt, scene, cull):
    name, S, _ = scene
    at = GOLDEN[name + "_occluded_cull"] == cull
    rays = np.ascontiguousarray(GOLDEN[name + "_occluded_rays"][at])
    dr, do = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(len(rays) * 4)
    S.occluded_device(dr.ptr, len(rays), do.ptr, cull=cull)
    assert np.array_equal(do.download(np.uint32, len(rays)), GOLDEN[name + "_occluded_ans"][at].ravel())
