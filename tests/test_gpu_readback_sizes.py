"""Read-backs at the sizes where their route changes: one chunk up to 16 KB, the
runtime's copy below 1.5 MB, the ring of three 4 MB chunks from there on, reused
past 12 MB and grown after a smaller read; against memory the runtime pinned."""
import ctypes

import numpy as np
import pytest
import torch

from cudapt_amd import scenes

pytestmark = pytest.mark.gpu


# counts take 4 bytes a pixel, images 12
@pytest.mark.parametrize("w,h", [(64, 64), (64, 65), (1365, 1), (1366, 1), (768, 511), (768, 512), (512, 255),
                                 (512, 256), (1024, 1025), (2048, 1025), (2048, 1537)])
def test_routes(cpt, w, h):
    sc = scenes.cornell()
    S = cpt.Scene(sc)
    R = cpt.Renderer(w, h, eye_depth=1, light_depth=1)
    R.render(S, sc["camera"], frames=2, result=False)
    for which, shape, dt in ((cpt.CPT_BUF_SAMPLE_N, (h, w), torch.int32), (cpt.CPT_BUF_RESULT, (h, w, 3), torch.float32),
                             (cpt.CPT_BUF_SAMPLE_N, (h, w), torch.int32)):
        pinned = torch.full(shape, -1, dtype=dt).pin_memory()
        assert cpt.lib().cpt_renderer_read_buffer(R.h, which, ctypes.c_void_p(pinned.data_ptr())) == 0
        want = pinned.numpy().view(np.uint32)
        assert np.array_equal(R.read(which).view(np.uint32), want)
        at = np.full(want.size + 9, 7, np.uint32)                    # nothing past the end
        assert cpt.lib().cpt_renderer_read_buffer(R.h, which, ctypes.c_void_p(at.ctypes.data + 4)) == 0
        assert np.array_equal(at[1:want.size + 1], want.ravel()) and at[0] == 7 and (at[want.size + 1:] == 7).all()
