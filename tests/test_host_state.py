"""The world's host state without a device: the C library is a stand-in that keeps the arrays it is given."""
import ctypes

import numpy as np
import pytest

from pe_amd import World, _abi
from pe_amd._abi import PeHipError

FIELDS = (("pos", 3), ("q", 4), ("v", 3), ("w", 3), ("normal", 3), ("d", 1))


class Library:
    """Bodies of one context.  A step moves every body and member by one in x and fails where told to."""

    def __init__(self):
        self.state, self.members, self.alive, self.fail, self.worlds = {}, None, 0, (), []

    def __getattr__(self, name):
        if not name.startswith("pehip_"):
            raise AttributeError(name)
        return lambda *a: 3 if name in self.fail else (getattr(self, "do_" + name[6:], lambda *b: 0)(*a) or 0)

    def pehip_last_error(self, ctx):
        return b"refused"

    def do_create(self, params, device, out):
        ctypes.cast(out, ctypes.POINTER(ctypes.c_void_p))[0] = 1
        self.alive += 1

    def do_destroy(self, ctx):
        self.alive -= 1

    def take(self, n, arrays):
        for (k, w), p in zip(FIELDS, arrays):
            self.state[k] = np.ctypeslib.as_array(p, (n, w)).copy()

    def do_upload_bodies(self, ctx, n, shape, sid, mat, fixed, param, pos, q, v, w, im, inertia, inverse, normal, d):
        self.take(n, (pos, q, v, w, normal, d))

    def do_upload_state(self, ctx, n, *arrays):
        before = self.state["pos"]
        self.take(n, arrays)
        if self.members is not None:                  # one union, the last body
            self.members = self.members + (self.state["pos"] - before)[-1]

    def do_download_state(self, ctx, n, *arrays):
        for (k, w), p in zip(FIELDS, arrays):
            np.ctypeslib.as_array(p, (n, w))[:] = self.state[k]

    def do_upload_members(self, ctx, k, owner, sid, mat, rad, rpos, gpos):
        given = np.ctypeslib.as_array(gpos, (k, 3))
        if not np.isfinite(given).all():
            return 1
        self.members = given.copy()

    def do_download_members(self, ctx, k, gpos):
        np.ctypeslib.as_array(gpos, (k, 3))[:] = self.members

    def do_step(self, ctx, dt, steps):
        for _ in range(steps):
            self.state["pos"][:, 0] += 1.0
            if self.members is not None:
                self.members[:, 0] += 1.0
        return 3 if "step" in self.fail else 0


@pytest.fixture
def lib(monkeypatch):
    library = Library()
    monkeypatch.setattr(_abi, "load", lambda: library)
    # the pointers stand for arrays of doubles
    monkeypatch.setattr("pe_amd.world.ptr", lambda a, typ=None: None if a is None else a.ctypes.data_as(
        ctypes.POINTER(np.ctypeslib.as_ctypes_type(a.dtype))))
    yield library
    for w in library.worlds:
        w._ctx = None                  # no handle of the stand-in's reaches the real library


def world(lib, union=False):
    w = World()
    lib.worlds.append(w)
    m = w.createMaterial("m", 1000.0, 0.0, 0.1, 0.1)
    w.createPlane(0, (0.0, 0.0, 1.0), 0.0, m)
    for k in range(3):
        w.createSphere(k + 1, (2.0 * k, 0.0, 1.0), 0.5, m)
    if union:
        w.createUnion(9, (0.0, 5.0, 1.0), [((0.0, 0.0, 0.0), 0.3, m), ((0.4, 0.0, 0.0), 0.3, m)])
    return w


def another(w, by):
    """Another state of the world, and a copy that no call has seen."""
    st = {k: v + by for k, v in w.getState().items()}
    return st, {k: v.copy() for k, v in st.items()}


def equal(a, b):
    for k, n in FIELDS:
        assert np.array_equal(np.reshape(a[k], (-1, n)), np.reshape(b[k], (-1, n))), k


def test_close_frees_the_context_whatever_fails(lib):
    w = world(lib)
    st, _ = another(w, 0.25)
    w.setState(st)
    lib.fail = ("pehip_download_state", "pehip_download_members")
    try:
        w.close()
    except PeHipError:
        pass
    assert lib.alive == 0 and w._ctx is None
    w.close()
    assert lib.alive == 0


def test_the_state_given_outlives_steps_and_the_context(lib):
    w = world(lib)
    st, given = another(w, 0.25)
    w.setState(st)
    for v in st.values():
        v += 1.0                       # the caller's arrays are the caller's
    w.run(3, 1e-3)
    w.close()                          # the steps' state was never asked for
    equal(w.host_arrays(), given)
    i = w.createSphere(9, (9.0, 9.0, 9.0), 0.5, 0)
    now = w.getState()                 # a new context, from the host's state
    equal({k: v[:i] for k, v in now.items()}, given)


def test_the_state_given_is_kept_where_a_run_fails_part_way(lib):
    w = world(lib)
    st, given = another(w, 0.25)
    w.setState(st)
    lib.fail = ("pehip_step",)
    lib.do_step(None, 0.0, 2)          # two steps were done
    with pytest.raises(PeHipError):
        w.run(4, 1e-3)
    equal(w.host_arrays(), given)


def test_a_held_dict_follows_and_keeps_what_is_written_into_it(lib):
    w = world(lib)
    held = w.host_arrays()
    before = held["pos"]
    kept = before.copy()
    st, given = another(w, 0.25)
    w.setState(st)
    equal(held, given)
    assert np.array_equal(before, kept)            # the array of before is not written over
    held["v"][1] = (1.0, 2.0, 3.0)
    given["v"][1] = (1.0, 2.0, 3.0)
    equal(w.host_arrays(), given)


def test_members_on_the_host_follow_the_state_given(lib):
    w = world(lib, union=True)
    st, given = another(w, 0.25)
    w.setState(st)
    st["mgpos"] += 1.0
    w.members()["gpos"][:] = 0.0
    assert np.array_equal(w.members()["gpos"], given["mgpos"])
    w.run(2, 1e-3)
    w.close()
    equal(w.host_arrays(), given)
    assert np.array_equal(w.members()["gpos"], given["mgpos"])
    w = world(lib, union=True)
    st, given = another(w, 0.25)
    del st["mgpos"]                                # the unions take their members along
    w.setState(st)
    assert np.array_equal(w.members()["gpos"], given["mgpos"])
    w.createMaterial("other", 1000.0, 0.0, 0.1, 0.1)
    assert np.array_equal(w.getState()["mgpos"], given["mgpos"])
    w.createUnion(10, (0.0, 9.0, 1.0), [((0.0, 0.0, 0.0), 0.3, 0)])
    assert np.array_equal(w.members()["gpos"][:2], given["mgpos"])


def test_the_state_given_is_the_hosts_where_its_members_are_refused(lib):
    w = world(lib, union=True)
    st, given = another(w, 0.25)
    st["mgpos"][1, 2] = np.nan
    with pytest.raises(PeHipError):
        w.setState(st)
    equal(w.host_arrays(), given)
    equal(w.getState(), given)
    w.setState(given)                              # and a good one is taken again
    assert np.array_equal(w.members()["gpos"], given["mgpos"])


def test_only_the_worlds_own_arrays_are_written_over(lib):
    made = world(lib).host_arrays()
    theirs = {k: v.copy() for k, v in made.items()}
    w = World()
    lib.worlds.append(w)
    w.createMaterial("m", 1000.0, 0.0, 0.1, 0.1)
    w.add_bodies(theirs)
    states = [another(w, 0.25 * k) for k in range(1, 5)]
    for st, given in states[:2]:
        w.setState(st)
    a = w.host_arrays()                            # from here on the arrays may be held
    equal(a, states[1][1])
    first = {k: a[k] for k, _ in FIELDS}
    w.setState(states[2][0])
    second = {k: a[k] for k, _ in FIELDS}
    w.run(1, 1e-3)
    w.host_arrays()
    w.setState(states[3][0])
    equal(a, states[3][1])
    equal(first, states[1][1])
    equal(second, states[2][1])
    equal(theirs, made)                            # what the bodies were made from
    for st, given in states:
        equal(st, given)                           # and the states given
    w.createSphere(9, (9.0, 9.0, 9.0), 0.5, 0)     # a new dict
    st, given = another(w, 1.0)
    w.setState(st)
    w.setState(given)
    equal(a, states[3][1])
    equal(w.host_arrays(), given)
