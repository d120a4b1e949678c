"""Small launches carry each path through every bounce in one kernel: images,
G-buffers, counts and ray statistics must be those of the bounce-by-bounce
passes, for batches whose waves carry 16 paths, some more, and 64."""
import numpy as np
import pytest

from cudapt_amd import scenes

pytestmark = pytest.mark.gpu

COUNTS = ("extension_rays", "shadow_rays", "eye_paths", "frames", "extend_nodes", "extend_tris", "shadow_nodes",
          "shadow_tris", "tail_rays", "tail_nodes", "tail_tris")


@pytest.fixture(scope="module")
def scene(cpt):
    sc = scenes.cornell()
    return sc, cpt.Scene(sc)


def _same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))


@pytest.mark.parametrize("w,h,frames,depth,fmt", [(1, 1, 1, 5, 1), (17, 3, 1, 1, 1), (129, 127, 2, 15, 1),
                                                  (419, 311, 1, 5, 1), (640, 360, 3, 5, 0), (1023, 513, 2, 5, 1)])
def test_plain(cpt, scene, w, h, frames, depth, fmt):
    sc, S = scene
    got, st = [], []
    for least in (0, 1 << 20):
        R = cpt.Renderer(w, h, eye_depth=depth, light_depth=3, **{
            "Frames In Flight": frames, "Refill Min Paths": least, "Node Format": fmt})
        got.append([R.render(S, sc["camera"], frames=frames) for _ in range(2)])
        s = R.stats()
        st.append([s[k] for k in COUNTS])
    _same(*got)
    assert st[0] == st[1]


@pytest.mark.parametrize("mode", ["PLL", "BINARY", "EMP"])
@pytest.mark.parametrize("w,h,tail", [(33, 17, 2), (200, 150, 1), (200, 150, 0)])
def test_adaptive(cpt, scene, mode, w, h, tail):
    sc, S = scene
    got, st = [], []
    for least in (0, 1 << 20):
        R = cpt.Renderer(w, h, mode=getattr(cpt, "CPT_MODE_BDPT_ADAPTIVE_" + mode), eye_depth=5, light_depth=3, **{
            "Refill Min Paths": least, "Tail Bounce": tail})
        img = [R.render(S, sc["camera"], frames=n) for n in (2, 3, 4)]
        got.append(img + [R.read(b) for b in (cpt.CPT_BUF_GBUF_POS, cpt.CPT_BUF_GBUF_NORM, cpt.CPT_BUF_GBUF_DIFF,
                                              cpt.CPT_BUF_ERROR, cpt.CPT_BUF_SAMPLE_N)])
        s = R.stats()
        st.append([s[k] for k in COUNTS])
    _same(*got)
    assert st[0][:4] == st[1][:4]
    # with a tail, bounces of the warm-up past it count as extension work where they are carried whole
    assert sum(st[0][4:8]) + sum(st[0][9:]) == sum(st[1][4:8]) + sum(st[1][9:])


@pytest.mark.parametrize("sizes,k", [([(5, 3)], 1), ([(64, 48), (33, 17), (100, 80)], 3)])
def test_views(cpt, scene, sizes, k):
    sc, S = scene
    got = []
    for pk in (64, 0):                              # a persistent extension grid keeps the passes
        views = [dict(sc["camera"], width=w, height=h) for w, h in sizes]
        B = cpt.Batch(views, frames_in_flight=k, eye_depth=5, light_depth=3)
        B.set_config(extend_chunk=pk)
        B.render(S, 2 * k)
        got.append([B.result(i) for i in range(len(sizes))])
    _same(*got)
