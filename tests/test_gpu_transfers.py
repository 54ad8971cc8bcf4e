"""Large copies go through pinned slots shared by several threads: bytes arrive whole at the edges of the pieces, at
unaligned host addresses, in pairs, from several threads at once (more than there are sets of slots), and after work
still running on the stream."""
import threading

import numpy as np
import pytest

from pypatools_amd import _lib
from pypatools_amd.device import DeviceArray, PinnedArray, to_host_pair

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


def _round_trip(n, offset, seed):
    src = np.random.default_rng(seed).integers(0, 256, n + offset, dtype=np.uint8)[offset:]
    d = DeviceArray((n,), np.uint8)
    _lib.call("pp_memcpy_h2d", d.ptr, src.ctypes.data, n, None)
    out = np.full(n + offset + 64, 7, np.uint8)
    _lib.call("pp_memcpy_d2h", out.ctypes.data + offset, d.ptr, n, None)
    assert np.array_equal(out[offset:offset + n], src)
    assert np.all(out[:offset] == 7) and np.all(out[offset + n:] == 7)


@pytest.mark.parametrize("offset", [0, 5])
@pytest.mark.parametrize("n", [1, 16383, 16384, 70001, MIB - 1, MIB, MIB + 1, 3 * MIB + 4095, 24 * MIB, 24 * MIB + 1, 32 * MIB - 1,
                               32 * MIB, 61 * MIB + 13])
def test_round_trip(n, offset):
    _round_trip(n, offset, n)


def test_pairs_after_running_work():
    a, b = DeviceArray((3, 700001)), DeviceArray((11,))
    for k in range(20):
        a.fill(float(k))
        b.fill(-float(k))
    ha, hb = to_host_pair(a, b)
    assert ha.shape == (3, 700001) and np.all(ha == 19.0) and np.all(hb == -19.0)


def test_several_threads():
    errors = []

    def work(k):
        try:
            for j in range(4):
                _round_trip(9 * MIB + 100 * k + j, k, 10 * k + j)
        except BaseException as e:      # noqa: BLE001 (handed to the test)
            errors.append(e)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors


def test_pinned_memory_and_release():
    p = PinnedArray(5 * MIB)
    v = p.view(np.uint8, 5 * MIB)
    v[:] = np.arange(5 * MIB, dtype=np.uint32).astype(np.uint8)
    d = DeviceArray((5 * MIB,), np.uint8)
    _lib.call("pp_memcpy_h2d", d.ptr, p.ptr, 5 * MIB, None)
    assert np.array_equal(d.to_host(), v)
    _lib.call("pp_release_staging")
    assert np.array_equal(d.to_host(), v)
