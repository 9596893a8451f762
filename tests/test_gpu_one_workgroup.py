"""Sweeps that run in one workgroup with their contacts on the chip, at the edges of what it holds.

Stacks of two spheres far apart, each with a floor contact and a sphere-sphere contact, give any number of
contacts.  The schedules all follow the same order of updates, so the states must agree bit for bit; the
adjoint's sweeps have no second schedule to choose, so a stack's gradient among many (in every one of the
adjoint's paths) is compared with that of the stack alone.
"""
import numpy as np
import pytest

from pe_amd import World, scenes
from pe_amd.adjoint import DifferentiableRun

pytestmark = pytest.mark.gpu

MATERIAL = [{"name": "m", "density": 1000.0, "cor": 0.0, "csf": 0.2, "cdf": 0.2}]


def stacks(contacts, model, sweeps, same=False):
    """Spheres with exactly `contacts` contacts: pairs, and one single sphere if odd.  same: every pair moves
    alike (the adjoint's comparison)."""
    rng = np.random.default_rng(contacts)
    pairs, single = contacts // 2, contacts % 2
    m = pairs + single
    side = int(np.ceil(np.sqrt(m)))
    at = 2.0 * np.stack([np.arange(m) % side, np.arange(m) // side], axis=1) + 1.0
    r = np.full(2 * m, 0.5)
    low = np.concatenate([at, np.full((m, 1), 0.5 - 1e-7)], axis=1)
    high = np.concatenate([at + [0.1, 0.05], np.full((m, 1), 0.5 + np.sqrt(1.0 - 0.0125) - 3e-7)], axis=1)
    pos = np.concatenate([low, high[:pairs]])
    r = r[:len(pos)]
    v = rng.uniform(-0.3, 0.3, size=(len(pos), 3))
    if same:
        one = rng.uniform(-0.05, 0.05, size=(2, 3))
        v = np.concatenate([np.repeat(one[:1], m, axis=0), np.repeat(one[1:], pairs, axis=0)])
    v[:, 2] = -0.05
    return scenes.Scene("stacks", MATERIAL, [((0, 0, 1), 0.0, 0)], pos, r, np.zeros(len(pos), np.uint32),
                        v0=np.concatenate([np.zeros((1, 3)), v]), dt=1e-3, max_iterations=sweeps, model=model)


def pairs(contacts, model, sweeps):
    """Falling pairs of spheres that touch: two bodies a contact."""
    rng = np.random.default_rng(contacts)
    side = int(np.ceil(np.sqrt(contacts)))
    at = np.stack([3.0 * (np.arange(contacts) % side), 3.0 * (np.arange(contacts) // side), np.full(contacts, 9.0)], axis=1)
    pos = np.concatenate([at, at + [0.6, 0.0, 0.8 - 1e-7]])
    v = rng.uniform(-0.3, 0.3, size=pos.shape)
    v[contacts:] -= [0.3, 0.0, 0.4]                  # the upper one comes nearer
    return scenes.Scene("pairs", MATERIAL, [((0, 0, 1), 0.0, 0)], pos, np.full(len(pos), 0.5),
                        np.zeros(len(pos), np.uint32), v0=np.concatenate([np.zeros((1, 3)), v]), dt=1e-3,
                        max_iterations=sweeps, model=model)


def step(scene, schedule, abort=0.0):
    w = World(device=0)
    scene.to_world(w)
    w.setSweepSchedule(schedule)
    w.setAbortThreshold(abort)
    w.simulationStep(scene.dt)
    out = w.getState(), w.impulses(), w.stats()
    w.close()
    return out


def same(a, b):
    for k in ("pos", "q", "v", "w"):
        assert np.array_equal(a[0][k], b[0][k]), k
    assert np.array_equal(a[1], b[1])
    assert a[2]["iterations"] == b[2]["iterations"] and a[2]["last_delta"] == b[2]["last_delta"]


# a lane, a wavefront, the register-held and the wide workgroup, and the schedule after them
@pytest.mark.parametrize("contacts", [1, 2, 63, 64, 65, 255, 256, 257, 511, 512, 513, 767, 768, 769])
@pytest.mark.parametrize("model,abort", [(0, 0.0), (1, 0.0), (1, 1e-4), (2, 0.0)])
def test_automatic_choice_equals_colour_launches(contacts, model, abort):
    sc = stacks(contacts, model, 20)
    a, b = step(sc, 0, abort), step(sc, 1, abort)
    assert a[2]["num_contacts"] == contacts
    assert (a[2]["schedule_used"] == 3) == (contacts <= 768)
    same(a, b)


# two bodies a contact fill the table of the bodies' places
@pytest.mark.parametrize("contacts", [256, 768])
@pytest.mark.parametrize("model", [0, 1, 2, 4])
def test_pairs_fill_the_workgroup(contacts, model):
    sc = pairs(contacts, model, 20)
    a, b = step(sc, 0), step(sc, 1)
    assert a[2]["num_contacts"] == contacts and a[2]["schedule_used"] == 3
    assert np.abs(a[1]).max() > 0
    same(a, b)


# the models with a search keep their schedules
@pytest.mark.parametrize("contacts", [1, 17, 256, 257])
@pytest.mark.parametrize("model", [3, 5])
def test_searching_models_keep_their_schedules(contacts, model):
    sc = stacks(contacts, model, 10)
    a, b, c = step(sc, 0), step(sc, 1), step(sc, 3)
    assert a[2]["schedule_used"] == 2 and c[2]["schedule_used"] == 3
    same(a, b)
    same(c, b)


def gradient(contacts, like=None):
    """Gradients of a run of contacts / 2 stacks; like: with the velocities that the stacks of so many contacts
    have."""
    sc = stacks(contacts, 1, 100, same=True)
    if like is not None:
        v = stacks(like, 1, 100, same=True).v0
        sc.v0[1:] = v[[1, 1 + like // 2]]
    run = DifferentiableRun(sc, 3, checkpoint_every=3, max_iterations=400, abort_threshold=1e-13, adjoint_sweeps=400,
                            adjoint_tol=1e-13)
    run.forward(sc.v0[1:], 0.4)
    pairs = contacts // 2
    weight = np.zeros((2 * pairs + 1, 3))
    weight[1:1 + pairs] = [1.0, -0.5, 0.25]
    weight[1 + pairs:] = [-0.75, 0.5, 1.0]
    g = run.backward(weight)
    assert run.last_stats["max_contacts"] == contacts
    run.close()
    return g, pairs


# held in registers (up to 512), from L2 (up to 550 a colour: the stacks have two), colour launches
@pytest.mark.parametrize("contacts", [510, 512, 514, 1100, 1102, 2048, 2050])
def test_adjoint_of_many_stacks_is_each_stacks_own(contacts):
    (gx, gv, gw, gmu), _ = gradient(2, like=contacts)
    (hx, hv, hw, hmu), pairs = gradient(contacts)
    for g, h in ((gx, hx), (gv, hv), (gw, hw)):
        for k in (0, 1):
            rows = h[1 + k * pairs:1 + (k + 1) * pairs]
            # the stacks differ by their place only: coordinates up to 70 with 1e-14 of rounding against
            # overlaps of 1e-7, and both runs converge to 1e-13
            assert np.max(np.abs(rows - g[1 + k])) <= 1e-6 * max(1.0, np.max(np.abs(g)))
    assert abs(hmu - pairs * gmu) <= 1e-6 * pairs * max(1.0, abs(gmu))


def towers(count, floating=0):
    """Towers of three spheres that lean, each with a floor contact, all alike, and free spheres above them."""
    side = int(np.ceil(np.sqrt(count)))
    at = 3.0 * np.stack([np.arange(count) % side, np.arange(count) // side], axis=1) + 1.0
    step_up = np.sqrt(1.0 - 0.0125) - 3e-7
    pos = np.concatenate([np.concatenate([at + [0.1 * k, 0.05 * k], np.full((count, 1), 0.5 - 1e-7 + k * step_up)], axis=1)
                          for k in range(3)])
    v = np.repeat(np.random.default_rng(5).uniform(-0.05, 0.05, size=(3, 3)), count, axis=0)
    v[:, 2] = -0.05
    k = np.arange(floating)
    free = np.stack([2.0 * (k % 64), 2.0 * (k // 64), np.full(floating, 20.0)], axis=1)
    pos, v = np.concatenate([pos, free]), np.concatenate([v, np.zeros((floating, 3))])
    return scenes.Scene("towers", MATERIAL, [((0, 0, 1), 0.0, 0)], pos, np.full(len(pos), 0.5),
                        np.zeros(len(pos), np.uint32), v0=np.concatenate([np.zeros((1, 3)), v]), dt=1e-3,
                        max_iterations=400, model=1)


def tower_gradient(count, floating=0):
    sc = towers(count, floating)
    run = DifferentiableRun(sc, 3, checkpoint_every=3, max_iterations=2000, abort_threshold=1e-13, adjoint_sweeps=2000,
                            adjoint_tol=1e-13)
    run.forward(sc.v0[1:], 0.4)
    weight = np.zeros((len(sc.v0), 3))
    for k, w in enumerate(([1.0, -0.5, 0.25], [-0.75, 0.5, 1.0], [0.5, 0.75, -1.0])):
        weight[1 + k * count:1 + (k + 1) * count] = w
    g = run.backward(weight)
    assert run.last_stats["max_contacts"] == 3 * count
    run.close()
    return [x[1:1 + 3 * count] for x in g[:3]], g[3]


# coupled contacts: held, from L2 for the bodies' sake (more than 2,048) or the contacts', colour launches
@pytest.mark.parametrize("count,floating", [(1, 2044), (1, 2045), (170, 0), (171, 0), (366, 0), (700, 0)])
def test_adjoint_of_towers_is_each_towers_own(count, floating):
    g, gmu = tower_gradient(1)
    h, hmu = tower_gradient(count, floating)
    for a, b in zip(g, h):
        for k in range(3):
            # as above: places of 1e-14 against overlaps of 1e-7, through three contacts one above the other
            assert np.max(np.abs(b[k * count:(k + 1) * count] - a[k])) <= 4e-6 * max(1.0, np.max(np.abs(a)))
    assert abs(hmu - count * gmu) <= 4e-6 * count * max(1.0, abs(gmu))
