"""Batched scenes at the edges of their kernels: as many contacts as threads, one fewer and one more (the sweeps'
place on the chip), few and many sliding contacts a colour (by wavefronts or by lanes), few scenes (the kernels
bounded for 256 threads, one wavefront a SIMD) and many (two wavefronts a SIMD).

512 threads take none of these paths: the sweeps run in global memory, one lane a contact.  Every path follows
the same order of updates, so the results must agree bit for bit.
"""
import numpy as np
import pytest

from pe_amd.batch import BatchWorld

from test_gpu_one_workgroup import pairs, stacks
from test_gpu_parity import box_scene, dense_scene, poly_scene

pytestmark = pytest.mark.gpu


def floating(scene, bodies):
    """The scene with free spheres above it, until it has so many bodies (its plane included)."""
    k = bodies - 1 - len(scene.sphere_r)
    side = int(np.ceil(np.sqrt(k)))
    at = np.stack([2.0 * (np.arange(k) % side), 2.0 * (np.arange(k) // side), np.full(k, 30.0)], axis=1)
    scene.sphere_pos = np.concatenate([scene.sphere_pos, at])
    scene.sphere_r = np.concatenate([scene.sphere_r, np.full(k, 0.5)])
    scene.sphere_mat = np.zeros(len(scene.sphere_r), np.uint32)
    scene.v0 = np.concatenate([scene.v0, np.zeros((k, 3))])
    return scene


def results(scenes, model, abort, tunings, steps=2):
    world = BatchWorld(scenes, max_iterations=12, relaxation_model=model, abort_threshold=abort)
    start = world.getState()
    out = []
    for threads, blocks in tunings:
        world.setTuning(threads=threads, blocks_per_cu=blocks, steps_per_launch=1, use_graph=0)
        world.setState(start)
        world.run(steps)
        stats = world.sceneStats()
        out.append((world.getState(), stats["contacts"], stats["iterations"]))
    world.close()
    return out


def same(out):
    for state, contacts, iterations in out[1:]:
        for k in ("pos", "q", "v", "w"):
            assert np.array_equal(state[k], out[0][0][k]), k
        assert np.array_equal(contacts, out[0][1]) and np.array_equal(iterations, out[0][2])


@pytest.mark.parametrize("abort", [0.0, 1e-4])
@pytest.mark.parametrize("model", [0, 1, 2, 3, 4, 5])
def test_few_scenes(model, abort):
    sizes = [1, 4, 10, 11, 20, 39, 40, 42, 63, 64, 65, 127, 128, 129, 255, 256, 257]
    scenes = [stacks(n, model, 12) for n in sizes] + [pairs(n, model, 12) for n in sizes]
    scenes += [dense_scene(), poly_scene(), box_scene()]
    out = results(scenes, model, abort, [(512, 2), (64, 8), (128, 4), (256, 2)])
    same(out)
    first = results(scenes, model, abort, [(64, 8)], steps=1)[0]
    assert np.array_equal(first[1][:2 * len(sizes)], 2 * sizes)


# more scenes than fit at one wavefront a SIMD, all of about the same size and, for model 3, of over 200 bodies
@pytest.mark.parametrize("model,threads,blocks", [(m, 256, 2) for m in range(6)] + [(1, 128, 4), (3, 128, 4), (1, 64, 8)])
def test_many_scenes(model, threads, blocks):
    sizes = [threads - 1, threads, threads + 1]
    scenes = [stacks(n, model, 12) for n in sizes]
    if threads == 128:
        scenes = [floating(sc, 208) for sc in scenes]
    count = 1100 if threads == 256 else (1600 if threads == 128 else 2400)
    out = results([scenes[k % 3] for k in range(count)], model, 0.0, [(512, 2), (threads, blocks)])
    same(out)
    for k in range(3):       # and a scene's result does not depend on the others
        n = len(scenes[k].sphere_r) + 1
        lo = sum(len(scenes[j].sphere_r) + 1 for j in range(k)) + (sum(len(s.sphere_r) + 1 for s in scenes) if k else 0)
        alone = results([scenes[k]], model, 0.0, [(threads, blocks)])[0][0]
        assert np.array_equal(out[1][0]["pos"][lo:lo + n], alone["pos"])
        assert np.array_equal(out[1][0]["v"][lo:lo + n], alone["v"])


# 64 threads keep their corrections behind the bodies' places, up to 2,560 bodies
@pytest.mark.parametrize("bodies", [2559, 2560, 2561, 4096])
def test_one_wavefront_and_many_bodies(bodies):
    same(results([floating(stacks(64, 1, 12), bodies)], 1, 0.0, [(512, 2), (64, 8), (256, 2)]))
