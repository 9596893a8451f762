"""The state a program sets is the world's: read back, after other changes to the world, and after it is closed."""
import numpy as np
import pytest

from pe_amd import World, scenes
from pe_amd.world import granular_particle_spheres

pytestmark = pytest.mark.gpu


def world():
    rng = np.random.default_rng(3)
    sc = scenes.drop_scene(3, 3, 2, r=0.4, seed=4)
    sc.unions = [(np.array([1.5 + 2.0 * k, 8.0, 3.0]), granular_particle_spheres(rng, 0.5, 0)) for k in range(3)]
    w = World(device=0)
    sc.to_world(w)
    return w


def moved(w, seed):
    rng = np.random.default_rng(seed)
    st = w.getState()
    n = len(st["pos"])
    st["pos"][6:] += rng.uniform(0.0, 0.1, size=(n - 6, 3))
    st["v"][6:] = rng.uniform(-1.0, 1.0, size=(n - 6, 3))
    q = rng.normal(size=(n - 6, 4))
    st["q"][6:] = q / np.sqrt((q * q).sum(1))[:, None]
    st["mgpos"] += rng.uniform(0.0, 0.01, size=st["mgpos"].shape)
    return st


def equal(a, b):
    for k in ("pos", "q", "v", "w", "normal", "d"):
        assert np.array_equal(a[k], b[k]), k


def test_the_given_state_stays_the_worlds():
    w = world()
    st = moved(w, 1)
    given = {k: v.copy() for k, v in st.items()}
    w.setState(st)
    for v in st.values():
        v += 1.0                                   # the caller's arrays are the caller's
    equal(w.getState(), given)
    equal(w.host_arrays(), given)
    assert np.array_equal(w.members()["gpos"], given["mgpos"])
    w.setState(given)
    w.createMaterial("other", 1000.0, 0.0, 0.1, 0.1)   # the bodies go to the device again
    equal(w.getState(), given)
    w.setState(given)
    i = w.createSphere(0, (5.0, 5.0, 20.0), 0.3, 0)
    now = w.getState()
    equal({k: now[k][:i] for k in given if k != "mgpos"}, {k: given[k] for k in given if k != "mgpos"})
    assert np.array_equal(now["mgpos"], given["mgpos"])
    w.close()
    w = world()
    w.setState(given)
    w.close()
    equal(w.host_arrays(), given)


def test_a_step_from_the_given_state_does_not_depend_on_how_it_got_there():
    a, b = world(), world()
    st = moved(a, 2)
    a.run(3, 1e-3)
    a.setState(st)                     # the rotation matrices follow the new orientations
    b.setState(st)
    a.run(4, 1e-3)
    b.run(4, 1e-3)
    equal(a.getState(), b.getState())
    # ... and equals a world whose bodies were uploaded in that state
    c = world()
    arrays = c.host_arrays()
    for k in ("pos", "q", "v", "w"):
        arrays[k][:] = st[k]
    c._m_gpos = list(st["mgpos"])
    c.run(4, 1e-3)
    equal(a.getState(), c.getState())
    assert np.array_equal(a.getState()["mgpos"], c.getState()["mgpos"])
