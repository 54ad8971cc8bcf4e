"""The field of a space-charge solve builds its map from the device copy of its grids: the same values as a Field made
from its host grids, also after the solver's next solve, and in copies of the field."""
import copy

import numpy as np
import pytest

import pypatools_amd as pa
from pypatools_amd.space_charge import SpaceChargeSolver

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


@pytest.mark.parametrize("cells", [(5, 4, 6), (17, 32, 9)])
def test_field_from_device_grids(cells):
    rng = np.random.default_rng(sum(cells))
    ext = (0.02, 0.03, 0.04)
    solver = SpaceChargeSolver(ext, cells)
    p = rng.normal(0, 3e-3, (501, 3))
    _, E = solver.solve(p, np.full(501, 1e-12))
    host = {a: E._field[a].values.copy() for a in "xyz"}
    twin = copy.deepcopy(E)
    _, other = solver.solve(-p, np.full(501, 3e-12))
    pts = rng.uniform(-0.015, 0.015, (777, 3))
    want = pa.Field.from_arrays(solver.grid(), host)(pts)
    for f in (E, twin, copy.copy(E)):
        np.testing.assert_array_equal(f(pts), want)
    assert not np.array_equal(other(pts), want)
    b = pa.Field.from_arrays(solver.grid(), {a: 0.1 * np.ones(cells) for a in "xyz"})
    push = pa.Pusher(pa.IonSpecies("proton"), "boris")
    v = np.full((777, 3), 1e6)
    for got, ref in zip(push.push_batch(pts, v, E, b, 1e-11),
                        push.push_batch(pts, v, pa.Field.from_arrays(solver.grid(), host), b, 1e-11)):
        np.testing.assert_array_equal(got, ref)
