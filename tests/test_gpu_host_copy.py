"""Results copied out of device memory (csrc/host_copy.hpp): sizes around the
single copy's limit (1 MiB), a thread's chunk (256 KiB), a flagged block (16
KiB) and a launch's half of the pinned memory (1 MiB, 8 MiB above 4 MiB), whole
rows and the first K columns of wider ones; every value must arrive."""
import numpy as np
import pytest

import kites_amd as K
from conftest import case

pytestmark = pytest.mark.gpu


def _edgeless(n):
    return K.DeviceGraph(K.HostGraph.from_csr(np.zeros(n + 1, np.uint32), np.zeros(0, np.uint32),
                                              np.zeros(0, np.uint32)))


@pytest.mark.parametrize("n", [1, 3, 4095, 4097, (1 << 18) - 1, 1 << 18, (1 << 18) + 1,
                               (1 << 18) + 4099, (1 << 19) + 1, (1 << 20) - 1,
                               (1 << 20) + 3, (1 << 21) - 1, (1 << 21) + 1,
                               (1 << 22) + 65539])
def test_values(n):
    case(f"values n={n}")
    d = _edgeless(n)
    for _ in range(3):     # the second and third calls reuse the pinned memory
        d.init("cc")       # every vertex's value is its own id
        assert np.array_equal(d.values(), np.arange(n, dtype=np.uint32))


@pytest.mark.parametrize("k", [1, 2, 3, 5, 57, 63, 64])
def test_columns(k):
    """Column j of a k-source run against the 64-source run's; 70,000 vertices:
    17.9 MB of rows, from one chunk (k = 1) to three halves of the pinned
    memory."""
    case(f"columns k={k}")
    h = K.HostGraph.erdos_renyi(70000, 200000, 3, wmin=1, wmax=9)
    d = K.DeviceGraph(h)
    src = np.random.default_rng(5).integers(0, 70000, 64).astype(np.uint32)
    full, _ = d.batch("sssp", src)
    part, _ = d.batch("sssp", src[:k])
    assert part.shape == (d.n, k) and np.array_equal(part, full[:, :k])
    src = np.concatenate([src, src[::-1], src, src])
    full, _ = d.bfs256(src)
    assert np.array_equal(full[:, :64], d.batch("bfs", src[:64])[0])
    part, _ = d.bfs256(src[:4 * k - 1])
    assert np.array_equal(part, full[:, :4 * k - 1])


def test_two_threads():
    """Two graphs copied out at once from two threads."""
    import threading
    case("two threads")
    sizes = [(1 << 21) + 77, (1 << 20) + 5]
    bad = []

    def go(n):
        d = _edgeless(n)
        want = np.arange(n, dtype=np.uint32)
        for _ in range(10):
            d.init("cc")
            if not np.array_equal(d.values(), want):
                bad.append(n)
    ts = [threading.Thread(target=go, args=(n,)) for n in sizes]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
