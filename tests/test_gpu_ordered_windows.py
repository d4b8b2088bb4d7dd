"""Ordered mode: in-lists that start beside a task window's boundary (448 edges)
and light lists that reach past it, bit for bit against the oracle."""
import numpy as np
import pytest

import kites_amd as K
from conftest import case
from oracle import liboracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("at", [383, 384, 385, 446, 447, 448, 449, 450, 511, 512, 513, 895, 896,
                                897, 1343, 1344, 1345])
@pytest.mark.parametrize("after", [1, 2, 63, 64, 65])
def test_list_starts_beside_a_window(at, after):
    case(f"in-list of {after} edges at edge {at}")
    degs = [64] * (at // 64) + ([at % 64] if at % 64 else []) + [after, 64, 1, 64, 33]
    n = len(degs) + 300
    rng = np.random.default_rng(at * 100 + after)
    R = np.zeros(n + 1, np.int64)
    R[1:len(degs) + 1] = np.cumsum(degs)
    R[len(degs) + 1:] = R[len(degs)]
    C = np.concatenate([np.sort(rng.integers(0, n, d)) for d in degs])
    h = K.HostGraph.from_csr(R.astype(np.uint32), C.astype(np.uint32), np.ones(len(C), np.uint32))
    R, C, _, oR, oC, _ = h.arrays()
    W = np.float32(1.0) / np.diff(oR.astype(np.int64)).astype(np.float32)[C]
    d = K.DeviceGraph(h)
    got, info = d.pagerank(damping=0.85, tol=1e-4)
    exp, it = O.ordered_pagerank(R, C, W, oR, oC, np.ones(n, np.float32), np.ones(n, np.uint8),
                                 base=np.float32(1.0) - np.float32(0.85), damp=0.85, tol=1e-4)
    d.close()
    assert info["iterations"] == it and np.array_equal(got.view(np.uint32), exp.view(np.uint32))
