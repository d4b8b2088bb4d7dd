"""Tiny push iterations on graphs of short out-lists (run_push_few and its
one-atomic close): out-degrees at the limit of 64 and beside it, frontiers that
cross the bound on a wave's staged entries, with and without near-far, against
the oracle.  persist=0 keeps the one-workgroup loop out of the way; the graphs
are larger than the small-graph limit and their runs longer than the 16
iterations that keep the full grid."""
import numpy as np
import pytest

import kites_amd as K
from conftest import case
from oracle import liboracle as O

pytestmark = pytest.mark.gpu


def _circulant(n, d, stride, seed):
    """Edges v -> v + 1 + k * stride (mod n), k < d, weights U[1, 50]; the last
    vertex has no out-edges."""
    v = np.arange(n - 1, dtype=np.int64)
    s = np.repeat(v, d)
    t = (s + 1 + np.tile(np.arange(d, dtype=np.int64) * stride, n - 1)) % n
    w = np.random.default_rng(seed).integers(1, 51, len(s))
    return K.HostGraph.from_edges(n, s.astype(np.uint32), t.astype(np.uint32), w.astype(np.uint32))


@pytest.mark.parametrize("n,d,stride", [(80000, 4, 1), (80000, 4, 190), (20000, 63, 1),
                                        (20000, 64, 1), (20000, 64, 17), (20000, 65, 1),
                                        (300000, 1, 1), (120000, 3, 700)])
def test_short_out_lists(n, d, stride):
    case(f"short out-lists n={n} d={d} stride={stride}")
    h = _circulant(n, d, stride, n + d)
    R, C, E, *_ = h.arrays()
    g = K.DeviceGraph(h)
    src = 5 if d > 1 else n - 400      # a path: only its end
    dist, lev = O.dijkstra(R, C, E, src), O.bfs(R, C, src)
    for kw in (dict(persist=0), dict(persist=0, tiny_grid=1), dict(persist=0, tiny_grid=65),
               dict()):
        got, info = g.solve("bfs", src, **kw)
        assert np.array_equal(got, lev), ("bfs", kw)
        got, info = g.solve("sssp", src, **kw)
        assert np.array_equal(got, dist), ("sssp", kw)
        for delta in (7, 120):
            got, _ = g.solve("sssp", src, delta=delta, **kw)
            assert np.array_equal(got, dist), ("sssp", delta, kw)
    assert info["iterations"] > 16
    g.solve("sssp", src, persist=0, keep_stats=True)
    st = g.stats()
    assert all(st[i]["in_count"] == st[i - 1]["count"] for i in range(1, len(st)))
