"""Pull iterations that run on fewer workgroups than their launch has, around the
two bounds (workgroups per compute unit; vertices and edges per workgroup), on
graphs whose launches are larger than that: thread-per-vertex pulls of settled
runs, edge-balanced pulls, the source-split ones, against the oracle."""
import numpy as np
import pytest

import kites_amd as K
from conftest import case
from oracle import liboracle as O

pytestmark = pytest.mark.gpu


# 1.8M, 2.3M, 2.8M and 4.5M vertices and edges: launches of 880 to 2,200
# workgroups, edge-balanced pulls of 880 (all), 1,024, 1,080 and 1,760
@pytest.mark.parametrize("scale,ef", [(17, 13), (17, 17), (18, 10), (18, 16)])
def test_pull_grid(scale, ef):
    case(f"pull grid scale={scale} ef={ef}")
    h = K.HostGraph.rmat(scale, ef, seed=scale + ef)
    R, C, E, *_ = h.arrays()
    src = int(np.bincount(C, minlength=h.n).argmax())
    want = {"bfs": O.bfs(R, C, src), "sssp": O.dijkstra(R, C, E, src),
            "widest": O.widest(R, C, E, src)}
    g = K.DeviceGraph(h)
    for algo, vals in want.items():
        for kw in (dict(), dict(sched="plain"), dict(sched="forced", forced_variant="pull_lb"),
                   dict(sched="forced", forced_variant="pull_t"),
                   dict(sched="forced", forced_variant="pull_lb", split_pull=True),
                   dict(sched="forced", forced_variant="pull_lb", grid=1333)):
            got, _ = g.solve(algo, src, **kw)
            assert np.array_equal(got, vals), (algo, kw)
