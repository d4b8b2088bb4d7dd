"""An error that an earlier call of the runtime left behind (and that was
reported there) is not reported again by a copy of results."""
import ctypes

import numpy as np
import pytest

import kites_amd as K
from conftest import case

pytestmark = pytest.mark.gpu


@pytest.fixture
def stale():
    hip = ctypes.CDLL("libamdhip64.so")

    def plant():
        assert hip.hipSetDevice(10000) != 0      # an invalid device: refused on the host

    yield plant
    hip.hipGetLastError()
    assert hip.hipPeekAtLastError() == 0


@pytest.mark.parametrize("n", [1000, (1 << 18) + 5, (1 << 20) + 3, (1 << 22) + 7])
def test_values_after_an_unrelated_error(stale, n):
    case(f"values n={n} after an unrelated error")
    d = K.DeviceGraph(K.HostGraph.from_csr(np.zeros(n + 1, np.uint32), np.zeros(0, np.uint32),
                                           np.zeros(0, np.uint32)))
    d.init("cc")
    stale()
    assert np.array_equal(d.values(), np.arange(n, dtype=np.uint32))
    d.close()
