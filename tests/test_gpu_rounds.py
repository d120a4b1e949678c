"""Allocation rounds, one launch each, against the oracle on the device's own error
map: one pixel, part of a workgroup, more workgroups than counters, last rounds
that keep more pixels than slots are left, and frames of several batches."""
import numpy as np
import pytest

import oracle
from cudapt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [2, 3])
@pytest.mark.parametrize("w,h,nd", [(1, 1, 5), (17, 13, 1), (17, 13, 40), (160, 129, 5), (257, 200, 3)])
def test_rounds(cpt, mode, w, h, nd):
    sc = scenes.cornell()
    S = cpt.Scene(sc)
    R = cpt.Renderer(w, h, mode=mode, eye_depth=4, light_depth=3, **{"Desired Max Sampling": nd})
    F = 5
    for f in range(3):
        R.render(S, sc["camera"], frames=F if f == 0 else 1)
        if f == 0:
            continue                                # the warm-up allocates nothing
        err, counts = R.read(cpt.CPT_BUF_ERROR), R.read(cpt.CPT_BUF_SAMPLE_COUNTS)
        want, _ = oracle.alloc_rounds(err, w * h, bisect=mode == 2, desired=w * h / nd, frame=F + f - 1)
        assert np.array_equal(counts.reshape(-1), np.asarray(want).reshape(-1))
