"""The whole-wavefront circle search of relaxation model 3 against the sequential one.

40,000 bodies that each touch only the floor give one colour of 40,000 contacts.  The colour launches
relax it with one lane a contact (a sequential search), the dataflow launch with one wavefront a contact
(predicted outcomes, checked): every bit of the new state must agree, whatever the number of steps, for
spheres (isotropic tangential block, ties) and tilted capsules (any block).
"""
import numpy as np
import pytest

from pe_amd import World, scenes

pytestmark = pytest.mark.gpu

N = 20000


def sliding_scene(seed):
    rng = np.random.default_rng(seed)
    side = 200
    x, y = np.meshgrid(2.0 * np.arange(side) + 1.0, 2.0 * np.arange(side) + 1.0)
    at = np.stack([x.reshape(-1), y.reshape(-1)], axis=1)
    assert len(at) == 2 * N
    sph, cap = at[0::2], at[1::2]
    r = rng.uniform(0.2, 0.5, size=N)
    depth = rng.uniform(0.0, 1e-4, size=N)
    spos = np.concatenate([sph, (r - depth)[:, None]], axis=1)
    cr, cl = rng.uniform(0.1, 0.2, size=N), rng.uniform(0.3, 0.6, size=N)
    # the axis (body x) turned about y by the tilt, then about z by the heading
    tilt, head = rng.uniform(0.3, 1.2, size=N), rng.uniform(0.0, 2 * np.pi, size=N)
    cy, sy, cz, sz = np.cos(tilt / 2), np.sin(tilt / 2), np.cos(head / 2), np.sin(head / 2)
    q = np.stack([cz * cy, -sz * sy, cz * sy, sz * cy], axis=1)
    low = 0.5 * cl * np.sin(tilt) + cr
    cpos = np.concatenate([cap, (low - depth)[:, None]], axis=1)
    v = rng.uniform(-1.0, 1.0, size=(2 * N, 3))
    v[:, 2] = -rng.uniform(0.0, 0.5, size=2 * N)
    v[::7, :2] *= 1e-3        # some stick, some slide by little
    return scenes.Scene("sliding", [{"name": "m", "density": 1000.0, "cor": 0.0, "csf": 0.2, "cdf": 0.2}],
                        [((0, 0, 1), 0.0, 0)], spos, r, np.zeros(N, np.uint32), capsule_pos=cpos, capsule_r=cr,
                        capsule_len=cl, capsule_q=q, capsule_mat=np.zeros(N, np.uint32),
                        v0=np.concatenate([np.zeros((1, 3)), v]), dt=1e-3, max_iterations=2)


@pytest.fixture(scope="module")
def scene():
    return sliding_scene(11)


def step(scene, schedule, max_sub, exact):
    w = World(device=0)
    scene.to_world(w)
    w.setSweepSchedule(schedule)
    w.setMaxSubIterations(max_sub)
    w.setExactTrig(exact)
    w.simulationStep(scene.dt)
    st = w.getState()
    c = w.contacts()
    p = w.impulses()
    w.close()
    return st, c, p


# steps around a triple, a fork round (9 and 11), a chain round (20), and beyond what is remembered
@pytest.mark.parametrize("max_sub", [0, 1, 2, 3, 8, 9, 10, 11, 12, 13, 18, 19, 20, 21, 29, 33, 80])
def test_wavefront_search_equals_sequential(scene, max_sub):
    a, c, p = step(scene, 1, max_sub, False)
    b, _, q = step(scene, 2, max_sub, False)
    assert len(c["dist"]) >= 2 * N           # every body touches the floor
    slip = np.hypot(p[:, 0], p[:, 1])
    assert np.count_nonzero(slip >= 0.399 * p[:, 2]) > N      # most contacts slide
    assert np.array_equal(p, q)
    for k in ("pos", "q", "v", "w"):
        assert np.array_equal(a[k], b[k]), k


def test_wavefront_search_equals_sequential_exact_trig(scene):
    a, _, p = step(scene, 1, 20, True)
    b, _, q = step(scene, 2, 20, True)
    assert np.array_equal(p, q)
    for k in ("pos", "q", "v", "w"):
        assert np.array_equal(a[k], b[k]), k
