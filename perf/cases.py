"""The work whose time is followed: time steps, detection, batches of scenes and differentiable runs,
through the calls a user's program makes (World, BatchWorld, DifferentiableRun).

A case is a dict of plain values.  ``prepare`` builds its scene from the seed and, where the state of
interest is a pile that has formed, pours it for a few steps first; the state it reaches there is the
checkpoint from which every pass starts.  ``run`` is one pass: the checkpoint restored, the steps, the
new state read back, as in rollouts, parameter studies and restarts.

Contacts are relaxed one after the other (Gauss-Seidel), so a step's result depends on the order of the
contacts, which is the library's own, and the sliding contacts' golden-section search is decided by last
bits: neither has a value that a plain evaluation of the model would give.  ``exact`` therefore covers
detection, whose points, normals, distances and friction are defined by the bodies alone.
"""
import math

import numpy as np

from pe_amd import scenes
from pe_amd.adjoint import DifferentiableRun
from pe_amd.batch import BatchWorld
from pe_amd.world import World, granular_particle_spheres

THRESHOLD = 1e-8     # contact threshold, and the margin of every bounding box


def listed():
    return [
        # A handful of bodies with the World's default model: an interactive scene or a unit test of a
        # user's program, where launches and latency are all there is.
        {"name": "few_spheres", "kind": "pour", "n": 27, "rmin": 0.5, "rmax": 0.5, "model": 1, "sweeps": 100,
         "steps": 20, "packed": 3, "lead": 150, "dt": 1e-3, "exact_trig": False},
        # The 1,000-sphere configuration as a formed pile: 100 sweeps, friction by decoupling.
        {"name": "pile_1k", "kind": "pour", "n": 1000, "rmin": 0.5, "rmax": 0.5, "model": 3, "sweeps": 100,
         "steps": 5, "packed": 10, "lead": 300, "dt": 1e-3, "exact_trig": False},
        # A parity run: correctly rounded trig reproduces the host libm's decisions.
        {"name": "pile_exact_3k", "kind": "pour", "n": 3001, "rmin": 0.25, "rmax": 0.5, "model": 3, "sweeps": 50,
         "steps": 3, "packed": 15, "lead": 200, "dt": 1e-3, "exact_trig": True},
        # Every shape pair with a contact routine: spheres, boxes and capsules against each other and planes.
        {"name": "mixed_4k", "kind": "mixed", "n": 4096, "boxes": 0.25, "capsules": 0.25, "model": 3, "sweeps": 50,
         "steps": 4, "packed": 16, "lead": 500, "dt": 5e-4},
        # Granular particles (unions of two to four spheres), several contacts per neighbour.
        {"name": "grains_5k", "kind": "grains", "n": 5000, "model": 3, "sweeps": 50, "steps": 3, "packed": 2,
         "lead": 400, "dt": 5e-4},
        # The headline: a polydisperse pile of 200,000 spheres, 50 sweeps, mostly falling bodies over a
        # packed bottom.
        {"name": "pile_200k", "kind": "pour", "n": 200000, "rmin": 0.25, "rmax": 0.5, "model": 3, "sweeps": 50,
         "steps": 6, "packed": 5, "lead": 500, "dt": 5e-4, "exact_trig": False},
        # The mixed-shape pour at scale: 5 % boxes, 30 sweeps, detection over many bodies.
        {"name": "hopper_400k", "kind": "mixed", "n": 400000, "boxes": 0.05, "capsules": 0.0, "model": 3,
         "sweeps": 30, "steps": 5, "packed": 3, "lead": 300, "dt": 5e-4},
        # A dense packing, beyond the size up to which all sweeps share one launch: every colour fills the chip.
        {"name": "packing_60k", "kind": "packing", "n": 60000, "model": 3, "sweeps": 50, "steps": 2, "dt": 1e-3},
        # Contact detection alone on a packed state (initialisation, checks of a checkpoint).
        {"name": "detect_250k", "kind": "detect", "n": 250007, "rmin": 0.45, "rmax": 0.5},
        # Many small worlds at once (parameter studies).
        {"name": "batch_small", "kind": "batch", "scenes": 1500, "lo": 40, "hi": 100, "model": 3, "sweeps": 40,
         "steps": 10, "lead": 200, "dt": 1e-3},
        # The batched configuration: scenes of 50 to 2,000 spheres.
        {"name": "batch_2k", "kind": "batch", "scenes": 640, "lo": 50, "hi": 2000, "model": 3, "sweeps": 40,
         "steps": 10, "lead": 200, "dt": 1e-3},
        # Forward and backward of a differentiable run, each step converged to a threshold.
        {"name": "adjoint_216", "kind": "adjoint", "side": 6, "model": 1, "steps": 8, "every": 4, "dt": 5e-4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pour", "pour", "pour", "mixed", "grains", "packing", "detect", "batch", "batch", "adjoint"])
    if kind == "pour":
        n = _log(rng, 27, 200000)
        return {"kind": kind, "n": n, "rmin": rng.choice([0.25, 0.35, 0.5]), "rmax": 0.5,
                "model": rng.choice([0, 1, 3, 3, 3, 5]),
                "sweeps": rng.randint(30, 50) if n > 2000 else rng.randint(30, 100), "steps": rng.randint(2, 5),
                "packed": rng.randint(2, 10) if n < 3000 else rng.randint(1, 4), "lead": rng.randint(100, 300),
                "dt": 5e-4 if n > 2000 else 1e-3,
                "exact_trig": n < 3000 and rng.random() < 0.2}
    if kind == "mixed":
        n = _log(rng, 64, 300000)
        return {"kind": kind, "n": n, "boxes": rng.choice([0.05, 0.25, 1.0]) if n < 5000 else 0.05,
                "capsules": rng.choice([0.0, 0.25]) if n < 5000 else 0.0, "model": rng.choice([1, 3, 3]),
                "sweeps": rng.randint(20, 50) if n < 50000 else rng.randint(20, 30), "steps": rng.randint(2, 4),
                "packed": rng.randint(1, 6) if n < 5000 else rng.randint(1, 2), "lead": rng.randint(100, 300),
                "dt": 5e-4}
    if kind == "grains":
        return {"kind": kind, "n": _log(rng, 100, 5000), "model": rng.choice([1, 3]), "sweeps": rng.randint(30, 50),
                "steps": rng.randint(2, 3), "packed": rng.randint(1, 4),
                "lead": rng.randint(150, 300), "dt": 5e-4}
    if kind == "packing":
        return {"kind": kind, "n": rng.randint(24000, 60000), "model": rng.choice([0, 1, 3, 3]),
                "sweeps": rng.randint(20, 50), "steps": rng.randint(1, 2), "dt": 1e-3}
    if kind == "detect":
        return {"kind": kind, "n": _log(rng, 500, 250000), "rmin": rng.choice([0.3, 0.45]), "rmax": 0.5}
    if kind == "batch":
        lo = _log(rng, 30, 300)
        hi = min(2000, lo * rng.randint(1, 8))
        return {"kind": kind, "scenes": max(2, min(1500, int(_log(rng, 3000, 300000) / (0.5 * (lo + hi))))),
                "lo": lo, "hi": hi, "model": rng.choice([1, 3, 3]), "sweeps": rng.randint(20, 40),
                "steps": rng.randint(4, 10), "lead": rng.randint(100, 200), "dt": 1e-3}
    return {"kind": "adjoint", "side": rng.randint(3, 6), "model": rng.choice([0, 1]), "steps": rng.randint(4, 8),
            "every": rng.randint(2, 4), "dt": 5e-4}


def _material(mu):
    return [{"name": "granular", "density": 2500.0, "cor": 0.0, "csf": mu / 2, "cdf": mu / 2}]


def _per_side(n):
    """Bodies along a side of a column about as high as wide."""
    return max(1, int(math.ceil(n ** (1.0 / 3.0) - 1e-9)))


def _sites(rng, n, spacing, z0, jitter):
    """n jittered lattice sites in a column, and the box they fill: (sites, side, height)."""
    per = _per_side(n)
    nz = (n + per * per - 1) // (per * per)
    pos = scenes.lattice(per, per, nz, spacing, (spacing / 2, spacing / 2, z0), jitter, rng, count=n)
    return pos, per * spacing, z0 + (nz + 4) * spacing


def _stacks(rng, reach, spacing, jitter, packed, gap):
    """Bodies that fit in balls of radius `reach` stacked on a lattice of columns: the lowest `packed` layers
    nearly touch, the ones above are `gap` apart.  Returns (positions, velocities, side, height): the packed
    layers stirred, the others falling at 6 m/s."""
    n = len(reach)
    per = _per_side(n)
    layer = per * per
    pos, side, _ = _sites(rng, n, spacing, 0.0, 0.0)
    pos[:, :2] += rng.uniform(-jitter, jitter, size=(n, 2))
    v = rng.uniform(-0.5, 0.5, size=(n, 3))
    top = np.zeros(layer)
    for k in range((n + layer - 1) // layer):
        r = reach[k * layer:(k + 1) * layer]
        rows = slice(k * layer, k * layer + len(r))
        top[:len(r)] += rng.uniform(0.0, 0.01, size=len(r)) + (0.0 if k < packed else gap)
        pos[rows, 2] = top[:len(r)] + r
        top[:len(r)] += 2.0 * r
        if k >= packed:
            v[rows, 2] -= 6.0
    return pos, v, side, float(top.max()) + 4.0


def _pour_scene(case, rng):
    """Spheres falling onto a pile whose lowest layers have packed."""
    n, rmax = case["n"], case["rmax"]
    r = rng.uniform(case["rmin"], rmax, size=n)
    pos, v, side, high = _stacks(rng, r, 2.04 * rmax, 0.015 * rmax, case["packed"], 0.3)
    return scenes.Scene("pour", _material(0.5), scenes.box_planes(side, side, high), pos, r, np.zeros(n, np.uint32),
                        v0=np.concatenate([np.zeros((6, 3)), v]), dt=case["dt"], max_iterations=case["sweeps"],
                        model=case["model"])


def _mixed_scene(case, rng):
    """Spheres, boxes and capsules, the kinds spread evenly, falling onto a pile whose lowest layers have packed."""
    n = case["n"]
    nb = int(round(n * min(case["boxes"], 1.0 - case["capsules"])))
    nc = min(int(round(n * case["capsules"])), n - nb)
    ns = n - nb - nc
    r = rng.uniform(0.2, 0.4, size=ns)
    edges = rng.uniform(0.3, 0.6, size=(nb, 3))
    cr, cl = rng.uniform(0.12, 0.25, size=nc), rng.uniform(0.2, 0.45, size=nc)
    order = rng.permutation(n)      # lattice site -> body
    reach = np.concatenate([r, 0.5 * np.sqrt((edges * edges).sum(1)), cr + 0.5 * cl])
    at, vs, side, high = _stacks(rng, reach[order], 1.06, 0.005, case["packed"], 0.3)
    pos, v = np.empty_like(at), np.empty_like(vs)
    pos[order], v[order] = at, vs
    return scenes.Scene("mixed", _material(0.6), scenes.box_planes(side, side, high), pos[:ns], r,
                        np.zeros(ns, np.uint32), box_pos=pos[ns:ns + nb], box_len=edges,
                        box_q=scenes.shoemake_quaternions(rng, nb), box_mat=np.zeros(nb, np.uint32),
                        capsule_pos=pos[ns + nb:], capsule_r=cr, capsule_len=cl,
                        capsule_q=scenes.shoemake_quaternions(rng, nc), capsule_mat=np.zeros(nc, np.uint32),
                        v0=np.concatenate([np.zeros((6, 3)), v]), dt=case["dt"], max_iterations=case["sweeps"],
                        model=case["model"])


def _grains_scene(case, rng):
    """Granular particles falling onto a pile of them: (scene, velocities; unions are created at rest)."""
    n = case["n"]
    pos, v, side, high = _stacks(rng, np.full(n, 0.48), 1.01, 0.005, case["packed"], 0.3)
    shapes = np.random.default_rng(n)      # the particles are the case's, their places and velocities the seed's
    unions = [(pos[k], granular_particle_spheres(shapes, 0.5, 0)) for k in range(n)]
    return scenes.Scene("grains", _material(0.5), scenes.box_planes(side, side, high), unions=unions, dt=case["dt"],
                        max_iterations=case["sweeps"], model=case["model"]), v


def _packing_scene(case, rng):
    """Equal spheres that all touch their lattice neighbours, moving slowly."""
    n = case["n"]
    pos, side, high = _sites(rng, n, 0.9999, 0.49995, 2e-5)
    return scenes.Scene("packing", _material(0.4), scenes.box_planes(side, side, high), pos, np.full(n, 0.5),
                        np.zeros(n, np.uint32),
                        v0=np.concatenate([np.zeros((6, 3)), rng.uniform(-0.05, 0.05, size=(n, 3))]), dt=case["dt"],
                        max_iterations=case["sweeps"], model=case["model"])


def _detect_scene(case, rng):
    """A packing that is the case's own (so that its contacts are as many for every seed), the box and all, at
    a place of the seed's choice."""
    n = case["n"]
    own = np.random.default_rng(n)
    pos, side, high = _sites(own, n, 0.96, 0.48, 0.02)
    r = own.uniform(case["rmin"], case["rmax"], size=n)
    shift = rng.uniform(-5.0, 5.0, size=3)
    planes = [(nrm, float(d + np.dot(nrm, shift)), mat) for nrm, d, mat in scenes.box_planes(side, side, high)]
    return scenes.Scene("detect", _material(0.4), planes, pos + shift, r, np.zeros(n, np.uint32),
                        v0=np.concatenate([np.zeros((6, 3)), rng.uniform(-0.5, 0.5, size=(n, 3))]))


def _batch_scenes(case, rng):
    m = case["scenes"]
    own = np.random.default_rng(m)         # the sizes are the case's
    sizes = np.rint(np.exp(own.uniform(math.log(case["lo"]), math.log(case["hi"]), size=m))).astype(int)
    mus = rng.uniform(0.2, 0.8, size=m)
    out = []
    for k in range(m):
        ns = int(sizes[k])
        pos = scenes.lattice(8, 8, (ns + 63) // 64, 1.1, (1.15, 1.15, 0.6), 0.05, rng, count=ns)
        v = rng.uniform(-0.5, 0.5, size=(ns, 3))
        v[:, 2] -= 5.0
        out.append(scenes.Scene("scene %d" % k, _material(float(mus[k])), scenes.box_planes(10.0, 10.0, 40.0), pos,
                                np.full(ns, 0.5), np.zeros(ns, np.uint32),
                                v0=np.concatenate([np.zeros((6, 3)), v]), dt=case["dt"],
                                max_iterations=case["sweeps"], model=case["model"]))
    return out, mus


def _adjoint_scene(case, rng):
    """A touching block of spheres that settles on the floor."""
    k = case["side"]
    pos = scenes.lattice(k, k, k, 0.8 - 2e-6, (0.41, 0.41, 0.4 - 1e-6), 2e-7, rng)
    ns = len(pos)
    v = rng.uniform(-0.02, 0.02, size=(ns, 3))
    v[:, 2] -= 0.2
    scene = scenes.Scene("block", _material(0.5), [((0, 0, 1), 0.0, 0)], pos, np.full(ns, 0.4),
                         np.zeros(ns, np.uint32), dt=case["dt"], steps=case["steps"])
    return scene, v


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "batch":
        scs, mus = _batch_scenes(case, rng)
        world = BatchWorld(scs, scene_friction=(mus, mus))
        world.run(case["lead"])
        return {"case": case, "batch": world, "start": world.getState()}
    if kind == "adjoint":
        scene, v0 = _adjoint_scene(case, rng)
        diff = DifferentiableRun(scene, case["steps"], checkpoint_every=case["every"], model=case["model"],
                                 max_iterations=2000, abort_threshold=1e-12, adjoint_sweeps=2000, adjoint_tol=1e-12)
        weight = rng.uniform(-1.0, 1.0, size=(len(v0) + 1, 3))
        return {"case": case, "diff": diff, "v0": v0, "mu": 0.5, "weight": weight}
    v = None
    if kind == "grains":
        scene, v = _grains_scene(case, rng)
    else:
        scene = {"pour": _pour_scene, "mixed": _mixed_scene, "packing": _packing_scene,
                 "detect": _detect_scene}[kind](case, rng)
    world = scene.to_world(World())
    world.setExactTrig(bool(case.get("exact_trig", False)))
    if v is not None:
        state = world.getState()
        state["v"][6:] = v
        world.setState(state)
    if case.get("lead"):
        world.run(case["lead"], case["dt"])
    return {"case": case, "world": world, "start": world.getState()}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        world = state["batch"]
        world.setState(state["start"])
        world.run(case["steps"])
        return world.getState()
    if kind == "adjoint":
        diff = state["diff"]
        final = diff.forward(state["v0"], state["mu"])
        dpos, dv, dw, dmu = diff.backward(state["weight"])
        return {"final": final, "dpos": dpos, "dv": dv, "dw": dw, "dmu": dmu}
    world = state["world"]
    if kind == "detect":
        return world.detect()
    world.setState(state["start"])
    world.run(case["steps"], case["dt"])
    return world.getState()


def _contacts_estimate(case):
    """About how many contacts a step of the case holds (counted on the listed cases' states)."""
    kind, n = case["kind"], case.get("n", 0)
    layer = float(n) ** (2.0 / 3.0)
    if kind in ("pour", "mixed", "grains"):
        return min(float(n), (0.35 if kind == "pour" else 0.2) * case["packed"] * layer)
    if kind == "packing":
        return 3.0 * n
    if kind == "detect":
        return 1.2 * n
    if kind == "batch":
        return 0.75 * case["scenes"] * 0.5 * (case["lo"] + case["hi"])
    return 2.0 * case["side"] ** 3


def work(case):
    """Bytes: every body's state (17 doubles) read and written once, or for detection the boxes and velocities
    read and the contacts written.  Flops: a relaxation is about 300 operations (two inertia products, the
    contact frame's transforms, a 3 x 3 solve), and every sweep of every step relaxes every contact once."""
    kind, nc = case["kind"], _contacts_estimate(case)
    if kind == "detect":
        return {"bytes": case["n"] * 8 * 13.0 + nc * 72.0, "flops": case["n"] * 200.0}
    if kind == "adjoint":
        # forward, its re-run and the reverse sweeps: a few hundred converging sweeps each
        return {"bytes": case["side"] ** 3 * 8 * 34.0, "flops": 3 * case["steps"] * 300.0 * nc * 300.0}
    n = case["scenes"] * 0.5 * (case["lo"] + case["hi"]) if kind == "batch" else case["n"]
    return {"bytes": n * 8 * 34.0, "flops": case["steps"] * case["sweeps"] * nc * 300.0}


def _pairs_in_library_order(x, r):
    """Sphere pairs closer than the threshold as rows (slot, rank, a, b) with a < b, and every sphere's slot: its
    place among the spheres sorted by (grid cell, index); rank orders a's partners by (cell offset, index).  The
    grid is the library's: one level, periodic power-of-two dimensions."""
    n = len(x)
    box = 2.0 * (r.max() + THRESHOLD)
    span = box * 1.001
    dims = []
    for k in range(3):
        cells = int(math.ceil((x[:, k].max() - x[:, k].min() + box) / span) + 2)
        p = 1
        while p < cells:
            p <<= 1
        dims.append(max(4, min(512, p)))
    limit = max(4096, 8 * n)
    while dims[0] * dims[1] * dims[2] > limit:
        k = 0
        if dims[1] > dims[k]:
            k = 1
        if dims[2] > dims[k]:
            k = 2
        if dims[k] <= 4:
            break
        dims[k] >>= 1
    cell = np.floor((x - (r + THRESHOLD)[:, None]) * (1.0 / span)).astype(np.int64)

    def bucket(c):
        return ((c[:, 2] & (dims[2] - 1)) * dims[1] + (c[:, 1] & (dims[1] - 1))) * dims[0] + (c[:, 0] & (dims[0] - 1))

    key = bucket(cell)
    order = np.argsort(key, kind="stable")
    start = np.searchsorted(key[order], np.arange(dims[0] * dims[1] * dims[2] + 1))
    slot = np.empty(n, np.int64)
    slot[order] = np.arange(n)
    found = []
    for o in range(27):
        nb = bucket(cell + np.array([o % 3 - 1, (o // 3) % 3 - 1, o // 9 - 1]))
        lo, hi = start[nb], start[nb + 1]
        for j in range(int((hi - lo).max())):
            a = np.flatnonzero(lo + j < hi)
            b = order[lo[a] + j]
            keep = b > a
            a, b = a[keep], b[keep]
            d = x[a] - x[b]
            near = np.sqrt((d * d).sum(1)) - r[a] - r[b] < THRESHOLD
            found.append(np.stack([slot[a[near]], np.full(near.sum(), o * n + j), a[near], b[near]], axis=1))
    return np.concatenate(found), slot


def exact(case, seed):
    """Detection's points, normals, distances and friction in 64 bits.  (The order of the contacts is the
    library's: by the first sphere's grid cell and index, then the partner's cell and index, then planes.)"""
    if case["kind"] != "detect":
        return None
    scene = _detect_scene(case, np.random.default_rng(seed))
    x, r = scene.sphere_pos, scene.sphere_r
    pairs, slot = _pairs_in_library_order(x, r)
    a, b = pairs[:, 2], pairs[:, 3]
    d = x[a] - x[b]
    length = np.sqrt((d * d).sum(1))
    dist = length - r[a] - r[b]
    normal = d / length[:, None]
    rows = [(pairs[:, 0], pairs[:, 1], x[b] + normal * (r[b] + 0.5 * dist)[:, None], normal, dist)]
    n = len(x)
    for k, (nrm, off, _) in enumerate(scene.planes):
        nrm = np.asarray(nrm, float)
        dist = x @ nrm - r - off
        s = np.flatnonzero(dist < THRESHOLD)
        rows.append((slot[s], np.full(len(s), 27 * n + k), x[s] - (r[s] + dist[s])[:, None] * nrm,
                     np.repeat(nrm[None], len(s), axis=0), dist[s]))
    order = np.lexsort((np.concatenate([q[1] for q in rows]), np.concatenate([q[0] for q in rows])))
    pos, normal, dist = (np.concatenate([q[k] for q in rows])[order] for k in (2, 3, 4))
    return {"b1": None, "b2": None, "pos": pos, "normal": normal, "dist": dist, "mu": np.full(len(dist), 0.4)}
