"""cpt_trace_counters counts the queries: closest hits visit what cpt_trace_cost says
of the same rays over the 8-wide nodes (with the answers of the FP32 nodes a few
are traced a second time), occlusion rays no more than that and at least a node
each, and a reset starts over."""
import numpy as np
import pytest

from cudapt_amd import scenes
from tests.helpers import random_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 65, 32769, 500000])        # a lane, waves in part, past the staging, refilled lanes
def test_queries_are_counted(cpt, n):
    S = cpt.Scene(scenes.sphere_grid(grid=16))
    rays = random_rays(n, [-30, 0.0, -30], [30, 6.0, 30], seed=n)
    dr, dh = cpt.DeviceBuffer.from_array(rays), cpt.DeviceBuffer(n * 16)
    nodes, tris = S.trace_cost(rays, layout=2).sum(0, dtype=np.uint64)
    assert nodes >= n
    S.counters(reset=True)
    S.trace_device(dr.ptr, n, dh.ptr, layout=2)
    assert S.counters(reset=True) == dict(nodes=int(nodes), tris=int(tris))
    for query in (lambda: S.trace(rays), lambda: S.trace_device(dr.ptr, n, dh.ptr, layout=0)):
        query()
        c = S.counters(reset=True)
        assert nodes <= c["nodes"] <= 1.01 * float(nodes) + 100 and tris <= c["tris"] <= 1.01 * float(tris) + 100
    S.occluded_device(dr.ptr, n, dh.ptr)
    c = S.counters()
    assert n <= c["nodes"] <= 1.01 * float(nodes) + 100 and c["tris"] <= 1.01 * float(tris) + 100
    S.occluded_device(dr.ptr, n, dh.ptr)
    assert S.counters(reset=True) == {k: 2 * v for k, v in c.items()}
    assert S.counters() == dict(nodes=0, tris=0)
