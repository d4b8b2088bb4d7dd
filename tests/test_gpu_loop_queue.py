"""The one-workgroup loop appends a vertex to its queue once, however many
threads lower it in the same iteration: layers of w vertices, each joined to
all of the next layer, so every vertex gets w equal (BFS) or unequal (SSSP)
candidates at once.  An iteration's queue is then exactly one layer."""
import numpy as np
import pytest

import kites_amd as K
from conftest import case
from oracle import liboracle as O

pytestmark = pytest.mark.gpu


def _layers(w, count, seed):
    a = np.arange(w, dtype=np.int64)
    s = np.repeat(a, w)[None, :] + w * np.arange(count - 1)[:, None]
    t = np.tile(a, w)[None, :] + w * np.arange(1, count)[:, None]
    s, t = s.ravel(), t.ravel()
    src = w * count              # one vertex in front of the first layer
    s = np.concatenate([np.full(w, src), s])
    t = np.concatenate([a, t])
    wt = np.random.default_rng(seed).integers(1, 4, len(s))
    return K.HostGraph.from_edges(src + 1, s.astype(np.uint32), t.astype(np.uint32),
                                  wt.astype(np.uint32)), src


@pytest.mark.parametrize("w", [8, 16, 31, 32, 45, 55, 64])
def test_a_vertex_enters_a_queue_once(w):
    count = 60
    h, src = _layers(w, count, w)
    R, C, E, *_ = h.arrays()
    d = K.DeviceGraph(h)
    case(f"loop queue of {w} x {w} edges")
    for _ in range(5):
        got, info = d.solve("bfs", src, persist=4096, keep_stats=True)
        assert np.array_equal(got, O.bfs(R, C, src))
        st = d.stats()
        loop = [x for x in st if x["variant"] == 11]
        assert len(loop) >= count - 17     # all after the first chunk of 16 launches
        assert [x["count"] for x in st[:count - 1]] == [w] * (count - 1)
        assert all(x["count"] * w == x["sum_outdeg"] for x in st[:count - 1])
    want = O.dijkstra(R, C, E, src)
    for kw in (dict(persist=4096), dict(delta=3)):
        got, _ = d.solve("sssp", src, keep_stats=True, **kw)
        assert np.array_equal(got, want)
        assert max(x["count"] for x in d.stats()) <= d.n
    d.close()


@pytest.mark.parametrize("persist", [True, 2047, 2048, 2049, 3024, 3025, 4096, 16384])
@pytest.mark.parametrize("delta", [0, 1 << 20])
def test_out_edge_limit_is_the_one_asked_for(persist, delta):
    """Queues of 55 x 55 = 3,025 out-edges: the loop runs them when the limit
    reaches that far.  Left at the default, plain runs stop at 2,048 and
    near-far runs at 4,096; 2,048 asked for is 2,048 in both."""
    h, src = _layers(55, 60, 1)
    d = K.DeviceGraph(h)
    case(f"loop limit {persist} delta {delta}")
    limit = (4096 if delta else 2048) if persist is True else min(int(persist), 4096)
    got, _ = d.solve("sssp", src, persist=persist, delta=delta, keep_stats=True)
    R, C, E, *_ = h.arrays()
    assert np.array_equal(got, O.dijkstra(R, C, E, src))
    st = d.stats()
    full = [b["variant"] == 11 for a, b in zip(st[20:], st[21:]) if a["sum_outdeg"] == 3025]
    assert len(full) >= 30 and all(f == (3025 <= limit) for f in full)
    d.close()
