"""Freed device blocks serve later allocations of their size class: work still running when a block is freed is over
before the block is handed out again, blocks in use are never shared, a block cannot be freed twice, and the kept ones
go back on request."""
import ctypes
import threading

import numpy as np
import pytest

from pypatools_amd import _lib
from pypatools_amd.device import DeviceArray, mem_info, synchronize

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


def test_running_work_ends_before_reuse():
    for k in range(8):
        a = DeviceArray((40 * MIB // 8,))
        for j in range(30):
            a.fill(float(j))            # still running when the block is freed
        a.free()
        b = DeviceArray((40 * MIB // 8,))
        b.fill(-1.0 - k)
        assert np.all(b.to_host() == -1.0 - k)


@pytest.mark.parametrize("nbytes", [1, 256, 257, 2048, 2049, 100001, MIB, MIB + 1, 256 * MIB, 256 * MIB + 1])
def test_blocks_in_use_are_apart(nbytes):
    held = [DeviceArray((nbytes,), np.uint8) for _ in range(3)]
    held[1].free()
    held[1] = DeviceArray((nbytes,), np.uint8)
    spans = sorted((h.ptr, h.ptr + nbytes) for h in held)
    assert all(x[1] <= y[0] for x, y in zip(spans, spans[1:]))


def test_double_free_is_refused():
    a = DeviceArray((1000,))
    p = a.ptr
    a.free()
    assert _lib.lib().pp_free(ctypes.c_void_p(p)) != 0


def test_release_and_bound():
    synchronize()
    _lib.call("pp_release_staging")
    before = mem_info()[0]
    blocks = [DeviceArray((200 * MIB,), np.uint8) for _ in range(8)]
    for b in blocks:
        b.free()
    assert mem_info()[0] >= before - 8 * MIB
    _lib.call("pp_release_staging")
    assert mem_info()[0] >= before - 8 * MIB


def test_threads():
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        for _ in range(25):
            n = int(rng.integers(1, 300000))
            v = np.full(n, float(k))
            d = DeviceArray.from_host(v)
            if not np.array_equal(d.to_host(), v):
                bad.append(k)
            d.free()
    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
