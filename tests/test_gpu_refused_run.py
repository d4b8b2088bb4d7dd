"""A run that is refused before it begins leaves the start in place: the next
run of any schedule begins from it, as if the refused call had not been made."""
import numpy as np
import pytest

import kites_amd as K
from conftest import case
from oracle import liboracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    h = K.HostGraph.rmat(12, 8, seed=4, wmin=1, wmax=63)
    R, C, E, oR, *_ = h.arrays()
    top = np.argsort(np.diff(oR.astype(np.int64)), kind="stable")[::-1].astype(np.uint32)
    return h, R, C, E, top


def _refuse(d, algo, how):
    with pytest.raises(K.KitesError):
        if how == "learned without a model":
            d.run(algo, sched="learned")
        else:
            d.record(algo, sched="learned")


@pytest.mark.parametrize("how", ["learned without a model", "recorder without a model"])
@pytest.mark.parametrize("algo", ["sssp", "bfs", "widest", "cc"])
def test_single_source(graph, algo, how):
    h, R, C, E, top = graph
    src = int(top[0])
    want = {"sssp": lambda: O.dijkstra(R, C, E, src), "bfs": lambda: O.bfs(R, C, src),
            "widest": lambda: O.widest(R, C, E, src),
            "cc": lambda: O.fixpoint(R, C, E, O.cc_init(len(R) - 1)[0], O.CC)[0]}[algo]()
    d = K.DeviceGraph(h)
    for kw in (dict(), dict(sched="classic"), dict(sched="forced", forced_variant="push_lb"),
               dict(sched="plain", gran=1)):
        case(f"{algo} after a refused run ({how}), then {kw}")
        d.init(algo, src)
        _refuse(d, algo, how)
        _refuse(d, algo, how)
        d.run(algo, **kw)
        assert np.array_equal(d.values(), want), kw
    d.close()


@pytest.mark.parametrize("algo", ["sssp", "bfs"])
def test_source_list(graph, algo):
    h, R, C, E, top = graph
    srcs = top[:70:3]
    one = (lambda s: O.dijkstra(R, C, E, int(s))) if algo == "sssp" else (lambda s: O.bfs(R, C, int(s)))
    want = np.minimum.reduce([one(s) for s in srcs])
    d = K.DeviceGraph(h)
    for kw in (dict(), dict(sched="classic"), dict(sched="forced", forced_variant="pull_lb")):
        case(f"{algo} from a list after a refused run, then {kw}")
        d.init_sources(algo, srcs)
        _refuse(d, algo, "learned without a model")
        d.run(algo, **kw)
        assert np.array_equal(d.values(), want), kw
    d.close()


def test_without_allocation(graph):
    """A refused call of the allocation-free entry point, which makes the
    start itself, leaves it to kites_graph_run."""
    h, R, C, E, top = graph
    src = int(top[1])
    d = K.DeviceGraph(h)
    case("refused allocation-free call, then a run")
    with pytest.raises(K.KitesError):
        d.sssp_noalloc(src, sched="learned")
    d.run("sssp")
    assert np.array_equal(d.values(), O.dijkstra(R, C, E, src))
    d.close()
