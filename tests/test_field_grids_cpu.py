"""Building the device map of a solve's field (its grids come with a device copy): which values it takes, what keeps
the copy alive while it is read, and what gives it back.  The map constructor is a stand-in, so nothing runs on a
device."""
import copy
import pickle
import threading

import numpy as np
import pytest

from pypatools_amd import engine, field
from pypatools_amd.field import Field

CELLS = (4, 3, 5)
N = 4 * 3 * 5


class Copy:
    """Stands for the (3, nodes) DeviceArray of the grids."""
    shape = (3, N)

    def __init__(self):
        self.freed = False
        self.ptr = 4096

    def view_ptr(self, offset):
        return self.ptr + 8 * offset

    def free(self):
        self.freed = True

    def __del__(self):
        self.freed = True


class Map:
    """Records what a device map is made from."""
    made = []

    def __init__(self, points, components, fill_value=0.0, periodic_z=False, **kw):
        self.points, self.components, self.kw = points, components, kw
        self.handle = id(self)
        self.from_device = not any(isinstance(c, np.ndarray) for c in components)
        Map.made.append(self)


@pytest.fixture
def solved(monkeypatch):
    """A field as a solve returns it."""
    Map.made = []
    monkeypatch.setattr(field, "DeviceFieldMap", Map)
    monkeypatch.setattr(engine, "DeviceFieldMap", Map)
    monkeypatch.setattr(engine, "_FUSED_CACHE", {})

    def make():
        axes = {a: np.linspace(-1.0, 1.0, n) for a, n in zip("xyz", CELLS)}
        E = Field.from_arrays(axes, {a: np.full(CELLS, float(k)) for k, a in enumerate("xyz")})
        dev = Copy()
        E._attach_device_grids(dev)
        return E, dev
    return make


def test_map_comes_from_the_device_copy_once(solved):
    E, _ = solved()
    m = E.device_map()
    assert m.from_device and E.device_map() is m and len(Map.made) == 1


def test_two_threads_make_one_map_from_a_living_copy(solved, monkeypatch):
    """The second thread enters device_map while the first is inside the constructor."""
    E, dev = solved()
    alive = dev.__dict__                    # outlives the copy itself
    del dev
    inside, entered, seen = threading.Event(), threading.Event(), []

    class Slow(Map):
        def __init__(self, *a, **k):
            super().__init__(*a, **k)
            inside.set()
            if len(Map.made) == 1:
                entered.wait(5)
            seen.append(alive["freed"])
    monkeypatch.setattr(field, "DeviceFieldMap", Slow)
    got, errors = [], []

    def work(first):
        try:
            if not first:
                inside.wait(5)
                threading.Timer(0.2, entered.set).start()
            got.append(E.device_map())
        except Exception as e:              # noqa: BLE001 - reported below
            errors.append(e)
    ts = [threading.Thread(target=work, args=(k == 0,)) for k in range(2)]
    [t.start() for t in ts]
    [t.join(10) for t in ts]
    assert not errors
    assert len(Map.made) == 1 and got[0] is got[1]
    assert seen == [False]                  # the copy was there until the constructor had returned


def test_copy_lives_until_the_constructor_returns(solved, monkeypatch):
    """A solve (or another user) that gives the copy back meanwhile does not free it under the reader."""
    E, dev = solved()
    alive = dev.__dict__
    del dev
    seen = []

    class Interrupted(Map):
        def __init__(self, *a, **k):
            E._drop_device_grids()
            seen.append(alive["freed"])
            super().__init__(*a, **k)
    monkeypatch.setattr(field, "DeviceFieldMap", Interrupted)
    E.device_map()
    assert seen == [False] and alive["freed"]


def _values(E, m):
    assert not m.from_device
    for k, c in enumerate("xyz"):
        np.testing.assert_array_equal(m.components[k], E._field[c].values)


def _edit_in_place(E):
    E._field["y"].values[1, 1, 1] = 7.0


def _rebind_values(E):
    E._field["z"].values = np.full(CELLS, 9.0)


def _keep_and_edit(E):
    kept = E._field["x"].values
    kept *= 3.0


def _replace_component(E):
    axes = {a: np.linspace(-1.0, 1.0, n) for a, n in zip("xyz", CELLS)}
    E._field["x"] = Field.from_arrays(axes, {a: np.full(CELLS, 5.0) for a in "xyz"})._field["x"]


def _replace_field(E):
    axes = {a: np.linspace(-1.0, 1.0, 2 * n) for a, n in zip("xyz", CELLS)}
    E._field = Field.from_arrays(axes, {a: np.ones([2 * n for n in CELLS]) for a in "xyz"})._field


@pytest.mark.parametrize("edit", [_edit_in_place, _rebind_values, _keep_and_edit, _replace_component, _replace_field])
def test_edited_host_grids_count(solved, edit):
    E, _ = solved()
    edit(E)
    _values(E, E.device_map())


def test_axes_of_another_length_do_not_take_the_copy(solved):
    """The map constructor reads as many values as the axes have nodes."""
    E, _ = solved()
    for c in "xyz":
        E._field[c].grid = tuple(np.linspace(-1.0, 1.0, 2 * n) for n in CELLS)
    assert not E.device_map().from_device


def test_a_fused_map_gives_the_copy_back(solved):
    E, dev = solved()
    axes = {a: np.linspace(-1.0, 1.0, n) for a, n in zip("xyz", CELLS)}
    B = Field.from_arrays(axes, {a: np.ones(CELLS) for a in "xyz"})
    alive = dev.__dict__
    del dev
    m = engine._fused_map(E, B)
    assert alive["freed"] and not m.from_device
    for k, c in enumerate("xyz"):
        np.testing.assert_array_equal(m.components[k], np.full(CELLS, float(k)))
    _values(E, E.device_map())


def test_fields_of_earlier_turns_hold_no_copy(solved, monkeypatch):
    """A program that keeps the field of every turn unevaluated keeps one device copy, not one per turn."""
    from pypatools_amd import space_charge
    copies = []

    class Dev(Copy):
        def __init__(self, shape, *a):
            super().__init__()
            self.shape, self.nbytes = shape, 8 * N
            if shape == (3, N):
                copies.append(self.__dict__)
    monkeypatch.setattr(space_charge, "DeviceArray", Dev)
    monkeypatch.setattr(space_charge._lib, "call", lambda *a: None)
    monkeypatch.setattr(space_charge, "to_host_pair", lambda a, b: (np.zeros(N), np.zeros(N)))
    s = space_charge.SpaceChargeSolver.__new__(space_charge.SpaceChargeSolver)
    s.cells, s.extent, s.n_dofs, s.turn_count = CELLS, (1.0, 1.0, 1.0), N, 0
    s.h = tuple(L / n for L, n in zip(s.extent, s.cells))
    s.phi, s.E = Dev((N,)), [Dev((N,)) for _ in range(3)]
    kept = [s._potential_and_field()[1] for _ in range(5)]
    assert [c["freed"] for c in copies] == [True] * 4 + [False]
    assert kept[-1].device_map().from_device and not kept[0].device_map().from_device


def test_copies_and_pickles_take_the_host_grids(solved):
    E, _ = solved()
    for twin in (copy.copy(E), copy.deepcopy(E), pickle.loads(pickle.dumps(E))):
        _values(twin, twin.device_map())


def test_fields_saved_before_device_copies_existed(solved):
    """A field whose saved state knows nothing of the device copy builds its map from its grids."""
    E, _ = solved()
    state = {k: v for k, v in E.__dict__.items() if "dev_values" not in k and "device_grids" not in k}
    old = Field.__new__(Field)
    old.__dict__.update(state)
    _values(old, old.device_map())
