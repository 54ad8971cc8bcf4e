"""Strict FP64 pushes through 3-D maps that are not the common form (uneven axes, offsets, a loss test) against the
oracle, bit for bit: lookups that start from the cell of the last one, particles on nodes and faces, outside the map,
and crossing several cells a step."""
import numpy as np
import pytest

import pypatools_amd as pa
from oracle.field import OField, OPeriodicZ, ORF, OScaled
from oracle.pusher import OraclePusher
from pypatools_amd.electrodes import TriangleElectrodes, box_mesh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


def _setup(n, uneven, periodic, seed=5):
    rng = np.random.default_rng(seed)
    ax = {"x": np.linspace(-6e-3, 6e-3, 13), "y": np.linspace(-5e-3, 5e-3, 2), "z": np.linspace(1e-3, 15e-3, 29)}
    if uneven:
        for a in "xz":
            d = ax[a][1] - ax[a][0]
            ax[a][1:-1] += rng.uniform(-0.45, 0.45, len(ax[a]) - 2) * d
    E = {a: 1e6 * rng.standard_normal((13, 2, 29)) for a in "xyz"}
    B = {a: 0.3 * rng.standard_normal((13, 2, 29)) for a in "xyz"}
    zlo, zhi = (-0.2, 0.3) if periodic else (0.0, 16e-3)
    r0 = rng.uniform([-7e-3, -6e-3, zlo], [7e-3, 6e-3, zhi], (n, 3))
    v0 = 2e7 * np.column_stack([0.1 * rng.standard_normal((n, 2)), 1 + 0.01 * rng.standard_normal(n)])
    v0[::3] *= -1.0
    # on nodes and faces, where the search decides between two cells
    k = np.arange(n)
    r0[k % 5 == 0, 0] = ax["x"][k[k % 5 == 0] % 13]
    r0[k % 7 == 0, 2] = ax["z"][k[k % 7 == 0] % 29]
    r0[k % 11 == 0, 1] = ax["y"][k[k % 11 == 0] % 2]
    return ax, E, B, r0, v0


@pytest.mark.parametrize("algorithm", ["boris", "rk4", "rk4_rel", "vay_rel", "yoshida", "boris_rel"])
@pytest.mark.parametrize("form", ["uneven", "uneven_periodic", "uneven_rf_offset", "offset", "mesh", "mesh_rf"])
def test_forms_match_the_oracle(form, algorithm):
    uneven, periodic, mesh = form != "offset", form == "uneven_periodic", form.startswith("mesh")
    # evenly spaced maps take the build of this test above the sizes of the one for few particles only
    n = 131 if uneven else (12289 if algorithm.startswith("rk4") else 4097)
    ax, E, B, r0, v0 = _setup(n, uneven, periodic)
    make = dict(periodic_z=periodic)
    e, b = (pa.Field.from_arrays(ax, f, **make) for f in (E, B))
    oe, ob = (OPeriodicZ(ax, f) if periodic else OField.from_arrays(ax, f) for f in (E, B))
    if "offset" in form:
        e, oe = pa.ScaledField(e, 0.7, 1e4), OScaled(oe, 0.7, 1e4)
        b, ob = pa.ScaledField(b, 1.2, -0.1), OScaled(ob, 1.2, -0.1)
    if "rf" in form:
        e, b = pa.RFField(e, 6e8, 0.4, "cos"), pa.RFField(b, 6e8, 0.4, "sin")
        oe, ob = ORF(oe, 6e8, 0.4, "cos"), ORF(ob, 6e8, 0.4, "sin")
    elec = TriangleElectrodes(*box_mesh((0.9, 0.9, 0.9), (1.0, 1.0, 1.0))) if mesh else None      # nothing meets it
    steps, dt, rec = (9, 2e-10, 3) if uneven else (4, 2e-10, 2)       # 4 mm a step
    rh, vh, _ = pa.Pusher(pa.IonSpecies("proton"), algorithm, electrode_assembly=elec).track_batch(
        r0, v0, e, b, steps, dt, rec)
    orh, ovh, _ = OraclePusher(pa.IonSpecies("proton").q_over_m, algorithm).track_batch(r0, v0, oe, ob, steps, dt, rec)
    np.testing.assert_array_equal(rh, orh)
    np.testing.assert_array_equal(vh, ovh)


@pytest.mark.parametrize("algorithm", ["boris", "rk4"])
def test_non_finite_particles_stay_alone_on_uneven_axes(algorithm):
    ax, E, B, r0, v0 = _setup(64, True, False)
    e, b = (pa.Field.from_arrays(ax, f) for f in (E, B))
    push = pa.Pusher(pa.IonSpecies("proton"), algorithm)
    want = push.track_batch(r0, v0, e, b, 6, 2e-11, 1)
    r1, v1 = r0.copy(), v0.copy()
    r1[9, 0], r1[20, 2], v1[33, 1], r1[50, 1] = np.nan, np.inf, -np.inf, -np.inf
    got = push.track_batch(r1, v1, e, b, 6, 2e-11, 1)
    keep = ~np.isin(np.arange(64), [9, 20, 33, 50])
    for g, w in zip(got[:2], want[:2]):
        np.testing.assert_array_equal(g[:, keep], w[:, keep])
    assert np.isnan(got[0][-1, 9]).any() and np.isinf(got[0][-1, 20, 2])
