"""Pushes through sums of fields evaluated inside the step loop (pp_push_sum), against the same sums evaluated
into (n, 3) arrays by the field algebra.  Strict FP64 is bit for bit the same; FP64-fast contracts products and
sums into FMAs (a few ulp per step over 40 steps, bounded at 1e-12 of the path); FP32-mixed does the same
operations on both routes and is held to the mode's 1e-6 of the path."""
import numpy as np
import pytest

from pypatools_amd.field import CompositeField, Field, RFField, ScaledField
from pypatools_amd.pusher import Pusher
from pypatools_amd.species import IonSpecies

pytestmark = pytest.mark.gpu


def fields(case):
    rng = np.random.default_rng(5)

    def grid(n, shift=0.0, warp=False):
        ax = {a: np.linspace(-0.02, 0.02, m) + shift for a, m in zip("xyz", n)}
        if warp:
            ax["y"] = ax["y"] + 2e-4 * np.sin(7 * np.arange(n[1]))
        return ax

    def make(ax, amp, **kw):
        return Field.from_arrays(ax, {c: amp * rng.standard_normal([len(a) for a in ax.values()]) for c in "xyz"}, **kw)
    ax = grid((12, 9, 14))
    E1, B1 = make(ax, 1e5), make(ax, 0.2)
    E2 = make(grid((7, 8, 6), 1e-3), 1e5, scaling=0.7)
    if case == "self":                      # external maps + self field on another grid
        return E1 + E2, B1
    if case == "three":                     # left-nested sum, weighted, B a sum too, uniform term
        return ((E1 + E2) + Field(dim=0, field={"x": 1e4, "y": -2e4, "z": 5e3})) - ScaledField(E1, 0.3, 10.0), \
            CompositeField([B1, Field.zero()], [1.5, 2.0])
    if case == "rf":
        w = 2 * np.pi * 1e8
        return RFField(E1, w, 0.3, "cos") + E2, CompositeField([RFField(B1, w, 0.3, "sin")], [1.0])
    if case == "warped":                    # non-uniform grid (strict only)
        return make(grid((12, 9, 14), warp=True), 1e5) + E2, B1
    raise ValueError(case)


class Arrays:
    """The same field through the generic route: a callable that hides the sum from the field compiler."""
    time_dependent = True

    def __init__(self, f):
        self.f = f

    def __call__(self, pts, t=None):
        from pypatools_amd.device import DeviceArray
        from pypatools_amd.field import evaluate_on_device
        return evaluate_on_device(self.f, DeviceArray.from_host(pts), len(pts), Arrays.precision, t).to_host()


@pytest.mark.parametrize("case,alg,precision,n", [
    ("self", "boris", "fp64", 1), ("self", "boris", "fp64", 65), ("self", "boris", "fp64", 5003),
    ("three", "vay_rel", "fp64", 255), ("three", "rk4", "fp64", 64), ("rf", "rk4_rel", "fp64", 100),
    ("rf", "vay", "fp64", 4097), ("warped", "yoshida", "fp64", 63),
    ("self", "boris", "fp64_fast", 300), ("three", "vay", "fp64_fast", 64), ("self", "boris", "fp32_mixed", 300),
    ("rf", "boris_rel", "fp32_mixed", 70), ("self", "rk4", "fp32_mixed", 50),
])
def test_summed_fields_match_the_array_route(case, alg, precision, n):
    E, B = fields(case)
    rng = np.random.default_rng(n)
    r0 = rng.uniform(-0.021, 0.021, (n, 3))          # some start outside the maps
    v0 = rng.normal(0, 3e6, (n, 3))
    p = Pusher(IonSpecies("proton"), alg, precision=precision)
    Arrays.precision = precision
    steps, dt = 40, 1e-10
    got = p.track_batch(r0, v0, E, B, steps, dt, 10, t0=1e-9)
    ref = p.track_batch(r0, v0, Arrays(E), Arrays(B), steps, dt, 10, t0=1e-9)
    one = p.push_batch(r0, v0, E, B, dt, t=1e-9)
    one_ref = p.push_batch(r0, v0, Arrays(E), Arrays(B), dt, t=1e-9)
    if precision == "fp64":
        for a, b in zip((*got[:2], *one), (*ref[:2], *one_ref)):
            assert np.array_equal(a, b)
    else:
        tol = 1e-12 if precision == "fp64_fast" else 1e-6
        path = np.abs(ref[1]).max() * steps * dt
        assert np.abs(got[0] - ref[0]).max() <= tol * path
        assert np.abs(one[0] - one_ref[0]).max() <= tol * path
    assert np.array_equal(got[2], ref[2])
