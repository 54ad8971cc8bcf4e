"""Strict FP64 launches of few particles run one particle per row of 16 lanes, larger ones a lane per particle.  Particles
do not interact, so each must end bit for bit where it ends in a launch of the other kind (which the parity tests hold
against the oracle): evenly spaced axes and axes whose nodes are off the even spacing (the guessed cell is then wrong for
many lanes), outside the map, and far outside the period of a periodic map."""
import numpy as np
import pytest

import pypatools_amd as pa

pytestmark = pytest.mark.gpu
LIMIT = {"rk4": 12288, "rk4_rel": 12288}        # others: 4096


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


def _setup(n, periodic, jitter, seed=23):
    rng = np.random.default_rng(seed)
    ax = {"x": np.linspace(-6e-3, 6e-3, 13), "y": np.linspace(-5e-3, 5e-3, 2), "z": np.linspace(1e-3, 15e-3, 15)}
    if jitter:
        for a in "xz":
            ax[a][1:-1] += rng.uniform(-0.2, 0.2, len(ax[a]) - 2) * 1e-3
    sh = (13, 2, 15)
    E = {a: 1e6 * rng.standard_normal(sh) for a in "xyz"}
    B = {a: 0.3 * rng.standard_normal(sh) for a in "xyz"}
    e, b = (pa.Field.from_arrays(ax, f, periodic_z=periodic) for f in (E, B))
    zlo, zhi = (-0.2, 0.3) if periodic else (0.0, 16e-3)
    r0 = rng.uniform([-7e-3, -6e-3, zlo], [7e-3, 6e-3, zhi], (n, 3))
    v0 = 2e7 * np.column_stack([0.1 * rng.standard_normal((n, 2)), 1 + 0.01 * rng.standard_normal(n)])
    return e, b, r0, v0


@pytest.mark.parametrize("rf", [False, True])
@pytest.mark.parametrize("jitter", [False, True])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("algorithm", ["boris", "vay", "rk4", "rk4_rel", "yoshida"])
def test_rows_and_lanes_agree(algorithm, periodic, jitter, rf):
    limit = LIMIT.get(algorithm, 4096)
    e, b, r0, v0 = _setup(limit + 1, periodic, jitter)
    e = 0.7 * e
    if rf:
        e, b = pa.RFField(e, 6e8, 0.4, "cos"), pa.RFField(b, 6e8, 0.4, "sin")
    push = pa.Pusher(pa.IonSpecies("proton"), algorithm)
    rl, vl, _ = push.track_batch(r0, v0, e, b, 12, 2e-11, 4)
    for pick in (slice(0, 1), slice(0, 5), slice(7, 106), slice(1, limit + 1)):
        rs, vs, _ = push.track_batch(r0[pick], v0[pick], e, b, 12, 2e-11, 4)
        np.testing.assert_array_equal(rs, rl[:, pick])
        np.testing.assert_array_equal(vs, vl[:, pick])


@pytest.mark.parametrize("periodic", [False, True])
def test_non_finite_particles_stay_alone(periodic):
    e, b, r0, v0 = _setup(9, periodic, False)
    r0[3, 2], v0[5, 0] = np.nan, np.inf
    push = pa.Pusher(pa.IonSpecies("proton"), "rk4")
    rl, vl, _ = push.track_batch(np.tile(r0, (1400, 1)), np.tile(v0, (1400, 1)), e, b, 5, 2e-11, 1)
    rs, vs, _ = push.track_batch(r0, v0, e, b, 5, 2e-11, 1)
    np.testing.assert_array_equal(rs, rl[:, :9])
    np.testing.assert_array_equal(vs, vl[:, :9])
