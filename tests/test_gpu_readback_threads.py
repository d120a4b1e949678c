"""Renderers share one pinned ring: images read by several threads at once, and by
renderers that come and go, are each renderer's own."""
import threading

import numpy as np
import pytest

from cudapt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(32, 32), (1024, 768), (1280, 1024)])     # one chunk, the ring, the ring reused
def test_reads_at_once(cpt, w, h):
    sc = scenes.cornell()
    scene = cpt.Scene(sc)
    R = [cpt.Renderer(w, h, eye_depth=1, light_depth=1, seed=k + 1) for k in range(4)]
    want = [r.render(scene, sc["camera"], frames=2) for r in R]
    assert not np.array_equal(want[0], want[1])
    bad = []

    def read(k):
        for _ in range(20):
            if not np.array_equal(R[k].read(cpt.CPT_BUF_RESULT).view(np.uint32), want[k].view(np.uint32)):
                bad.append(k)

    threads = [threading.Thread(target=read, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_renderers_come_and_go(cpt):
    sc = scenes.cornell()
    scene = cpt.Scene(sc)
    images = []
    for _ in range(3):
        r = cpt.Renderer(800, 600, eye_depth=1, light_depth=1)
        images.append(r.render(scene, sc["camera"]))
        del r                                                # the last one: the ring goes with it
    assert all(np.array_equal(i, images[0]) for i in images)
