"""push and push_batch of up to 8192 particles hand their rows to the device through mapped host memory, larger batches
through device arrays: the same particles must end at the same bits either way, from several threads at once too."""
import threading

import numpy as np
import pytest

import pypatools_amd as pa

pytestmark = pytest.mark.gpu
MAX = 8192


@pytest.fixture(scope="module", autouse=True)
def _device():
    from pypatools_amd import device
    if device.device_count() == 0:
        pytest.skip("no HIP device visible")


def _fields(kind):
    rng = np.random.default_rng(3)
    if kind == "uniform":
        return (pa.Field(dim=0, field={"x": 1e4, "y": -2e4, "z": 3e4}), pa.Field(dim=0, field={"x": 0.1, "y": 0.0, "z": 0.9}))
    ax = {"x": np.linspace(-6e-3, 6e-3, 9), "y": np.linspace(-5e-3, 5e-3, 8), "z": np.linspace(0.0, 14e-3, 11)}
    e, b = (pa.Field.from_arrays(ax, {a: s * rng.standard_normal((9, 8, 11)) for a in "xyz"}) for s in (1e6, 0.4))
    if kind == "rf":
        e, b = pa.RFField(e, 6e8, 0.4, "cos"), pa.RFField(b, 6e8, 0.4, "sin")
    return e, b


def _particles(n):
    rng = np.random.default_rng(4)
    r = rng.uniform([-7e-3, -6e-3, -1e-3], [7e-3, 6e-3, 15e-3], (n, 3))
    return r, 3e7 * rng.standard_normal((n, 3))


@pytest.mark.parametrize("kind", ["uniform", "map", "rf"])
@pytest.mark.parametrize("algorithm", ["boris", "vay", "boris_rel", "rk4_rel"])
@pytest.mark.parametrize("precision", ["fp64", "fp64_fast", "fp32_mixed"])
def test_rows_and_arrays_agree(precision, algorithm, kind):
    e, b = _fields(kind)
    r, v = _particles(MAX + 1)
    push = pa.Pusher(pa.IonSpecies("proton"), algorithm, precision=precision)
    rl, vl = push.push_batch(r, v, e, b, 2e-11, t=1e-9)
    for pick in (slice(0, 1), slice(3, 68), slice(1, MAX + 1)):
        rs, vs = push.push_batch(r[pick], v[pick], e, b, 2e-11, t=1e-9)
        np.testing.assert_array_equal(rs, rl[pick])
        np.testing.assert_array_equal(vs, vl[pick])


def test_threads():
    e, b = _fields("map")
    r, v = _particles(600)
    push = pa.Pusher(pa.IonSpecies("proton"), "boris")
    want = push.push_batch(r, v, e, b, 2e-11)
    bad = []

    def work(k):
        for j in range(20):
            lo = 10 * k + j
            got = push.push_batch(r[lo:lo + 300], v[lo:lo + 300], e, b, 2e-11)
            if not all(np.array_equal(g, w[lo:lo + 300]) for g, w in zip(got, want)):
                bad.append(k)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
