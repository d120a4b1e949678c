"""Images read back in chunks through the pinned ring, at sizes around one chunk
and around the whole ring, against a direct copy to memory the runtime pinned."""
import ctypes

import numpy as np
import pytest
import torch

from cudapt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (512, 512), (513, 511), (1024, 1024), (1024, 1025), (1361, 257)])
def test_ring(cpt, w, h):
    sc = scenes.cornell()
    S = cpt.Scene(sc)
    R = cpt.Renderer(w, h, eye_depth=2, light_depth=2)
    img = R.render(S, sc["camera"], frames=2)
    for which, shape, dt in ((cpt.CPT_BUF_RESULT, (h, w, 3), torch.float32), (cpt.CPT_BUF_SAMPLE_N, (h, w), torch.int32)):
        pinned = torch.full(shape, -1, dtype=dt).pin_memory()
        assert cpt.lib().cpt_renderer_read_buffer(R.h, which, ctypes.c_void_p(pinned.data_ptr())) == 0
        got = R.read(which)
        assert np.array_equal(got.view(np.uint32), pinned.numpy().view(np.uint32))
        if which == cpt.CPT_BUF_RESULT:
            assert np.array_equal(got.view(np.uint32), img.view(np.uint32))
