"""The grid option: grids of the whole chip and more take the path that the
default takes on small graphs (captured chunks of small launches), so that no
shape the tuner tries is slower than the default for the launches' sake; smaller
grids are taken literally.  Same values with every grid."""
import numpy as np
import pytest

import kites_amd as K
from conftest import case
from oracle import liboracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algo", ["sssp", "bfs", "widest"])
def test_large_grids_on_a_small_graph(algo):
    h = K.HostGraph.rmat(9, 8, seed=5, wmin=1, wmax=255)
    R, C, E, oR, *_ = h.arrays()
    src = int(np.argmax(np.diff(oR.astype(np.int64))))
    want = {"sssp": O.dijkstra, "widest": O.widest}.get(algo, lambda r, c, e, s: O.bfs(r, c, s))(
        R, C, E, src)
    for per_cu in (1, 2, 14, 24, 28, 42):
        case(f"{algo} with {per_cu} workgroups per CU on 512 vertices")
        d = K.DeviceGraph(h)
        got, info = d.solve(algo, src, sched="plain", grid=256 * per_cu)
        assert np.array_equal(got, want)
        if per_cu >= 24:
            assert info["iterations"] < 16 and info["graph_builds"] == 1
            # the default run replays the same captured chunk
            got, info = d.solve(algo, src, sched="plain")
            assert np.array_equal(got, want) and info["graph_builds"] == 1
        d.close()


def test_tuned_options_on_a_small_graph():
    h = K.HostGraph.rmat(9, 8, seed=6, wmin=1, wmax=255)
    R, C, E, oR, *_ = h.arrays()
    src = int(np.argmax(np.diff(oR.astype(np.int64))))
    d = K.DeviceGraph(h)
    case("tuner on 512 vertices")
    best, ms, table = d.autotune("sssp", [src], sched="plain")
    assert len(table) == 24
    got, _ = d.solve("sssp", src, sched="plain", **best)
    assert np.array_equal(got, O.dijkstra(R, C, E, src))
    d.close()
