"""Rays with a negative eps, or so short that the box test's shift of small
components leads them off their triangles: queries answer as the FP32 4-wide
nodes do.  The rays and those answers (closest hit, occlusion flag) were
recorded from a kernel that traversed those nodes alone."""
import os

import numpy as np
import pytest

from cudapt_amd import scenes

pytestmark = pytest.mark.gpu

GOLDEN = np.load(os.path.join(os.path.dirname(__file__), "golden", "odd_rays.npz"))


@pytest.mark.parametrize("cull", [0, 1])
@pytest.mark.parametrize("name", ["grid", "cornell"])
def test_recorded_answers(cpt, name, cull):
    S = cpt.Scene(scenes.sphere_grid(grid=16) if name == "grid" else scenes.cornell())
    rays, want = GOLDEN[f"{name}_{cull}_rays"], GOLDEN[f"{name}_{cull}_ans"]
    n = len(rays)
    assert np.array_equal(S.trace(rays, cull=bool(cull)).view(np.uint32).reshape(-1, 4), want[:, :4])
    dr, do = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(n * 16)
    S.trace_device(dr.ptr, n, do.ptr, layout=0, cull=bool(cull))
    assert np.array_equal(do.download(np.uint32, n * 4).reshape(-1, 4), want[:, :4])
    S.occluded_device(dr.ptr, n, do.ptr, cull=bool(cull))
    assert np.array_equal(do.download(np.uint32, n), want[:, 4])
