"""The routes of a gather give the same bits: launches up to 131072 particles gather per lane, larger ones stage the
cells of a wavefront in LDS.  Particles do not interact, so a few of them tracked alone take the first route and
must end bit for bit where they end within a large launch."""
import numpy as np
import pytest

import pypatools_amd as pa
from pypatools_amd.batch import BatchedTracker, Bunch

pytestmark = pytest.mark.gpu
LIMIT = 131072


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


def _setup(n, periodic, seed=17):
    rng = np.random.default_rng(seed)
    ax = {"x": np.linspace(-6e-3, 6e-3, 13), "y": np.linspace(-5e-3, 5e-3, 11), "z": np.linspace(0.0, 14e-3, 15)}
    sh = (13, 11, 15)
    E = {a: 1e6 * rng.standard_normal(sh) for a in "xyz"}
    B = {a: 0.3 * rng.standard_normal(sh) for a in "xyz"}
    e, b = (pa.Field.from_arrays(ax, f, periodic_z=periodic) for f in (E, B))
    r0 = rng.uniform([-7e-3, -6e-3, -1e-3], [7e-3, 6e-3, 15e-3], (n, 3))     # some outside the map
    v0 = 2e7 * np.column_stack([0.1 * rng.standard_normal((n, 2)), 1 + 0.01 * rng.standard_normal(n)])
    return e, b, r0, v0


@pytest.mark.parametrize("rf", [False, True])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("algorithm", ["boris", "rk4_rel"])
@pytest.mark.parametrize("precision", ["fp32_mixed", "fp64_fast"])
def test_small_and_large_launches_agree(precision, algorithm, periodic, rf):
    e, b, r0, v0 = _setup(LIMIT + 1, periodic)
    if rf:
        e, b = pa.RFField(e, 6e8, 0.4, "cos"), pa.RFField(b, 6e8, 0.4, "sin")
    push = pa.Pusher(pa.IonSpecies("proton"), algorithm, precision=precision)
    rl, vl, _ = push.track_batch(r0, v0, e, b, 25, 2e-11, 5)
    for pick in (slice(0, 1), slice(0, 65), slice(1, LIMIT + 1)):
        rs, vs, _ = push.track_batch(r0[pick], v0[pick], e, b, 25, 2e-11, 5)
        np.testing.assert_array_equal(rs, rl[:, pick])
        np.testing.assert_array_equal(vs, vl[:, pick])


def test_small_and_large_batches_agree():
    e, b, r0, v0 = _setup(LIMIT + 200, True)
    def bunches(m):
        return [Bunch(r0[:m], v0[:m], 9.58e7, "boris", 30, 2e-11, 0.7, 1.3),
                Bunch(r0[-200:], v0[-200:], 4.8e7, "vay", 20, 2e-11)]
    def run(m):
        t = BatchedTracker([(e, b)])
        t.load(bunches(m)).run()
        return t.results()
    large, small = run(LIMIT), run(999)
    for q in (0, 1):
        np.testing.assert_array_equal(small[0][q], large[0][q][:999])
        np.testing.assert_array_equal(small[1][q], large[1][q])
