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
