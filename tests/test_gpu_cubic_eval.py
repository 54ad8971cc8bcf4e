"""The register-tap evaluation of 3-D cubic splines against scipy's map_coordinates (order 3, constant 0 outside, after
np.interp coordinates): the smallest grids it takes, uneven axes, one and three components, points on the faces.  Both
sum 64 products of weights whose absolute values add to 1: 1e-13 of the largest coefficient covers their rounding."""
import numpy as np
import pytest
from scipy.ndimage import map_coordinates

import pypatools_amd as pa
from pypatools_amd.interpolators import get_interpolator

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


@pytest.mark.parametrize("uneven", [False, True])
@pytest.mark.parametrize("shape", [(3, 3, 3), (2, 5, 7), (4, 3, 17), (13, 11, 9)])
def test_cubic_matches_map_coordinates(shape, uneven):
    rng = np.random.default_rng(sum(shape))
    axes = [np.linspace(-1.0, 2.0, n) for n in shape]
    if uneven:
        axes = [np.sort(a + np.r_[0.0, rng.uniform(-0.4, 0.4, len(a) - 2) * 3.0 / (len(a) - 1), 0.0]) for a in axes]
    vals = {c: rng.standard_normal(shape) for c in "xyz"}
    pts = np.concatenate([rng.uniform(-1.2, 2.2, (1003, 3)), np.array(np.meshgrid(*[a[[0, -1]] for a in axes])).reshape(3, -1).T,
                          np.column_stack([a[rng.integers(len(a), size=40)] for a in axes])])
    coords = [np.interp(pts[:, k], a, np.arange(len(a)), left=-1, right=len(a)) for k, a in enumerate(axes)]
    got = pa.Field.from_arrays(dict(zip("xyz", axes)), vals, method="cubic")(pts)
    for k, c in enumerate("xyz"):
        want = map_coordinates(vals[c], coords, order=3, mode="constant", cval=0.0)
        np.testing.assert_allclose(got[:, k], want, rtol=0, atol=3e-13 * 27)
        one = get_interpolator(tuple(axes), vals[c], method="cubic", fill_value=0.0)(pts)
        np.testing.assert_array_equal(one, got[:, k])
