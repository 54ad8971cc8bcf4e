"""Maps whose values go up in several pieces (more than 256 MiB) and whose layout kernel loops: every node holds its
value, and a periodic axis repeats its first node."""
import numpy as np
import pytest

from pypatools_amd import _lib
from pypatools_amd.device import DeviceArray
from pypatools_amd.interpolators import DeviceFieldMap, eval_term

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


@pytest.mark.parametrize("shape,periodic", [((7, 1021, 1601), False), ((7, 1021, 1601), True), ((3, 5, 4), True)])
def test_nodes_hold_their_values(shape, periodic):
    rng = np.random.default_rng(shape[2])
    vals = [rng.standard_normal(shape) for _ in range(3)]
    ax = [np.arange(n, dtype=np.float64) for n in shape]
    m = DeviceFieldMap(ax, vals, periodic_z=periodic, coefficients=False)
    term = _lib.PPField()
    term.kind, term.map, term.scale1 = _lib.FIELD_MAP, m.handle, 1.0
    n = 200000
    k = np.column_stack([rng.integers(0, s, n) for s in shape])
    k[:8] = [[x, y, z] for x in (0, shape[0] - 1) for y in (0, shape[1] - 1) for z in (0, shape[2] - 1)]
    pts = k.astype(np.float64)
    if periodic:
        pts[::2, 2] += shape[2]             # the same nodes one period on
    got = eval_term(term, DeviceArray.from_host(pts), n, "fp64").to_host()
    np.testing.assert_array_equal(got, np.column_stack([v[k[:, 0], k[:, 1], k[:, 2]] for v in vals]))
