"""Host logic of the engine's step loops, with the library calls replaced by stand-ins (no device)."""
import types

import numpy as np

from pypatools_amd import engine


def test_lossy_loop_reports_the_particles_that_are_left(monkeypatch):
    """active: the caller's mask of live particles, as the device left it (the benchmark's lost fraction)."""
    left = np.array([1, 0, 1, 1, 0], dtype=np.uint8)
    st = types.SimpleNamespace(n=5, alive=types.SimpleNamespace(ptr=0, to_host=lambda: left), unsort=lambda: None)
    calls = []
    monkeypatch.setattr(engine._lib, "call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(engine.Tracker, "_args", lambda self, *a, **k: types.SimpleNamespace())
    active = np.ones(5, dtype=bool)
    tr = engine.Tracker("boris", "fp64", 1.0, sort_every=0)
    tr._lossy_loop(st, None, 3, 1e-11, None, None, types.SimpleNamespace(handle=0), active, None, False)
    assert calls and set(calls) == {"pp_push_lossy"}
    np.testing.assert_array_equal(active, left.astype(bool))


def test_last_velocity_record_of_lost_particles(monkeypatch):
    """Resynchronised velocities overwrite the last record: of every particle in a track without a mask in its result
    (batch=False), of the live ones otherwise."""
    class Dev:
        def __init__(self, shape=(1,), dtype=np.float64):
            self.shape, self.nbytes, self.ptr = shape, 8, 4096

        @classmethod
        def from_host(cls, a):
            return cls(a.shape)

        def fill(self, v):
            pass
    st = types.SimpleNamespace(n=2, alive=None, vx=Dev(), vy=Dev(), vz=Dev(), positions_aos=lambda out: out)
    monkeypatch.setattr(engine, "DeviceArray", Dev)
    monkeypatch.setattr(engine, "FieldPair", lambda e, b: types.SimpleNamespace(direct=True, time_dependent=False))
    monkeypatch.setattr(engine.ParticleState, "from_host", classmethod(lambda cls, r, v: st))
    monkeypatch.setattr(engine, "to_host_pair", lambda a, b: (None, None))
    monkeypatch.setattr(engine.Tracker, "_kick", lambda *a: None)
    monkeypatch.setattr(engine.Tracker, "_slow_loop", lambda *a: None)
    masks = []
    monkeypatch.setattr(engine._lib, "call", lambda name, *a: masks.append(a[3]) if name == "pp_velocity_rows" else 0)
    tr = engine.Tracker("boris", "fp64", 1.0)
    for batch in (True, False):
        tr.track(np.zeros((2, 3)), np.ones((2, 3)), None, None, 4, 1e-11, 2, batch=batch, electrode_assembly=object())
    assert masks == [None, 4096, None, None]        # record 0 and the last one of either call


def test_sums_with_time_dependent_members_of_other_kinds_keep_the_array_route():
    """A member that declares itself time dependent without being an RFField has no factor for the push kernels; a sum
    with one is evaluated term by term, as before the sums moved into the step loop."""
    from pypatools_amd.field import Field, RFField, compile_sum
    const = {"x": 1.0, "y": 0.0, "z": 2.0}
    drifting = Field(dim=0, field=const)
    drifting.time_dependent = True
    plain, rf = Field(dim=0, field=const), RFField(Field(dim=0, field=const), 1e8)
    assert compile_sum(plain + plain, plain) is not None
    assert compile_sum(plain + rf, plain) is not None
    assert compile_sum(plain + drifting, plain) is None
    assert compile_sum(rf + drifting, plain) is None
    assert compile_sum(plain + plain, 2.0 * drifting) is None
    fp = engine.FieldPair(plain + drifting, plain)
    assert not fp.fused("boris", "fp64") and not fp.direct
