"""The dealing of rays to the refilling waves at its edges: fewer rays than waves,
up to one chunk of 64 a wave and just past it, shares that differ in length, and
chunks that shrink towards a share's end.  One workgroup a compute unit, so that
few rays reach each case; images and ray counts must be those of one ray a thread."""
import numpy as np
import pytest

from cudapt_amd import scenes

pytestmark = pytest.mark.gpu

# 1,024 waves on 256 compute units: 65,536 rays are dealt once, 65,537 in shares
SIZES = [(1, 1, 1), (63, 65, 1), (128, 129, 2), (256, 256, 1), (65537, 1, 1), (511, 129, 3), (640, 360, 8)]


@pytest.fixture(scope="module")
def scene(cpt):
    sc = scenes.cornell()
    return sc, cpt.Scene(sc)


@pytest.mark.parametrize("w,h,frames", SIZES)
def test_dealt_rays(cpt, scene, w, h, frames):
    sc, S = scene
    got = []
    for refill in (0, 16):
        R = cpt.Renderer(w, h, eye_depth=4, light_depth=3, **{
            "Frames In Flight": frames, "Refill Min Paths": 0, "Refill Workgroups": 1, "Traversal Refill": refill,
            "Secondary Refill": refill, "Shadow Refill": refill})
        for _ in range(2):                          # the counters start again at zero
            img = R.render(S, sc["camera"], frames=frames)
        st = R.stats()
        got.append((img.copy(), st["extension_rays"], st["shadow_rays"], st["extend_nodes"], st["shadow_nodes"]))
    a, b = got
    assert np.array_equal(a[0].view(np.uint32), b[0].view(np.uint32))
    assert a[1:] == b[1:]
