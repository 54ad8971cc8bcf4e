"""Arguments of the device map as they reach the library (a stand-in), no device."""
import ctypes

import numpy as np
import pytest

from pypatools_amd import interpolators
from pypatools_amd.interpolators import DeviceFieldMap


@pytest.fixture
def calls(monkeypatch):
    made = []

    def call(name, parts, on_device, ncomp, nx, ny, nz, gx, gy, gz, fill, flags, out):
        n = nx * ny * nz
        made.append((on_device, [parts[c] if on_device else
                                 list((ctypes.c_double * n).from_address(parts[c])) for c in range(ncomp)]))
    monkeypatch.setattr(interpolators._lib, "call", call)
    return made


@pytest.mark.parametrize("components", [[3, 4, 5], [3, 4.0, 5], [True, False, 2], [np.int64(3), 4, 5], [[3], [4], [5]]])
def test_whole_numbers_are_values(calls, components):
    """A one-node map of whole numbers holds these numbers, not what lies at such an address."""
    DeviceFieldMap([[0.0], [0.0], [0.0]], components)
    want = [[float(np.asarray(c).reshape(()) if np.ndim(c) == 0 else c[0])] for c in components]
    assert calls == [(0, want)]


def test_addresses_are_named(calls):
    DeviceFieldMap([[0.0, 1.0]], [4096, 8192, 12288], on_device=True)
    assert calls == [(1, [4096, 8192, 12288])]


def test_no_components(calls):
    DeviceFieldMap([[0.0, 1.0]], [])
    assert calls == [(0, [])]                   # refused by the library
