"""Ordered mode at the edges of its work split (detail/ordered_kernel.hpp):
in-lists around 64 edges (one chunk, the light limit) and of the other lengths
up to 512 and beyond, in several orders (so that lists start all over a task's
window of 448 edges), with vertices without in-edges between them; the values and the iteration count must be the oracle's bit for
bit (the combine order is defined, so no tolerance)."""
import numpy as np
import pytest

import kites_amd as K
from conftest import case
from oracle import liboracle as O

pytestmark = pytest.mark.gpu

DEGREES = [1, 2, 3, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 319, 320,
           321, 511, 512, 513, 767, 768, 769, 1000, 4097]


def _graph(degs, n, seed):
    """n vertices, the first len(degs) with these in-degrees, sources drawn
    uniformly (repeats and self-loops kept), weights 1."""
    rng = np.random.default_rng(seed)
    deg = np.zeros(n, np.int64)
    deg[:len(degs)] = degs
    R = np.concatenate([[0], np.cumsum(deg)])
    C = rng.integers(0, n, R[-1])
    for v in range(len(degs)):
        C[R[v]:R[v + 1]].sort()
    return K.HostGraph.from_csr(R.astype(np.uint32), C.astype(np.uint32),
                                np.ones(len(C), np.uint32))


def _check(h, damping, tol):
    R, C, _, oR, oC, _ = h.arrays()
    n = len(R) - 1
    outdeg = np.diff(oR.astype(np.int64)).astype(np.float32)
    W = np.float32(1.0) / outdeg[C]
    got, info = K.DeviceGraph(h).pagerank(damping=damping, tol=tol)
    exp, it = O.ordered_pagerank(R, C, W, oR, oC, np.ones(n, np.float32), np.ones(n, np.uint8),
                                 base=np.float32(1.0) - np.float32(damping), damp=damping, tol=tol)
    assert it > 0 and info["iterations"] == it
    assert np.array_equal(got.view(np.uint32), exp.view(np.uint32)), \
        f"differ at {np.flatnonzero(got != exp)[:10]}"


@pytest.mark.parametrize("order", ["ascending", "descending", "shuffled", "gaps"])
def test_ordered_in_list_lengths(order):
    case(f"ordered in-list lengths {order}")
    degs = list(DEGREES)
    if order == "descending":
        degs.reverse()
    elif order == "shuffled":
        np.random.default_rng(3).shuffle(degs)
    elif order == "gaps":
        # runs of vertices without in-edges and of single-edge ones between
        degs = [x for d in degs for x in [d] + [0] * (d % 130) + [1] * (d % 7)]
    _check(_graph(degs, max(len(degs), 700) + 37, 5), 0.85, 0.0)


@pytest.mark.parametrize("tol", [0.0, 1e-3])
def test_ordered_few_movers(tol):
    """A dense core feeding a long path: after the core settles only the path
    moves, so iterations change from testing every edge's source to walking
    the movers' out-lists."""
    case(f"ordered few movers tol {tol}")
    rng = np.random.default_rng(9)
    core, path = 300, 500
    src = [rng.integers(0, core, 20000), np.arange(core - 1, core + path - 1)]
    dst = [rng.integers(0, core, 20000), np.arange(core, core + path)]
    s, d = np.concatenate(src), np.concatenate(dst)
    h = K.HostGraph.from_edges(core + path, s.astype(np.uint32), d.astype(np.uint32),
                               np.ones(len(s), np.uint32))
    _check(h, 0.9, tol)
