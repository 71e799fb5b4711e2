"""Scenes of 1e8 to 2e12 units (at 1e13 a hit's t overflows), whose node sizes times the reciprocal of a direction component near zero pass the range of
FP32: rays along the axes, in the triangles' planes and with components down to 1e-30 find what brute force finds, by
quads and by lanes, alone and in a batch with a small scene."""
import numpy as np
import pytest

import eleven
from test_gpu_slabs import both_ways


def boxes(rng):
    """Axis-aligned grids on the faces of nested cubes, and triangles of any direction."""
    i, j = (a.ravel() for a in np.meshgrid(np.arange(6), np.arange(6)))
    faces = []
    for half in (1.0, 0.4):
        at = lambda a, b, z: np.stack([(a / 3 - 1) * half, (b / 3 - 1) * half, np.full(len(a), z)], -1)  # noqa: E731
        for z in (-half, half):
            g = np.concatenate([np.stack([at(i, j, z), at(i + 1, j, z), at(i + 1, j + 1, z)], 1),
                                np.stack([at(i, j, z), at(i + 1, j + 1, z), at(i, j + 1, z)], 1)])
            faces += [np.roll(g, k, axis=2) for k in range(3)]
    return np.concatenate(faces + [rng.uniform(-1, 1, (200, 1, 3)) + rng.normal(scale=0.1, size=(200, 3, 3))])


@pytest.mark.gpu
@pytest.mark.parametrize("size", [1e8, 1e10, 1e11, 1e12, 2e12])
@pytest.mark.parametrize("kind", ["axes", "two axes", "small components"])
def test_components_near_zero(gpu_ctx, size, kind):
    print(f"[large scenes] {size:g}, {kind}", flush=True)
    rng = np.random.default_rng(3)
    v = (boxes(rng) * size).astype(np.float32).reshape(-1, 9)
    n = 2048
    o = rng.uniform(-1.5, 1.5, (n, 3))
    d = rng.normal(size=(n, 3))
    if kind == "axes":
        d = np.eye(3)[rng.integers(0, 3, n)] * rng.choice([-1.0, 1.0], (n, 1))
    elif kind == "two axes":
        d[np.arange(n), rng.integers(0, 3, n)] = rng.choice([0.0, -0.0], n)
    else:
        d[np.arange(n), rng.integers(0, 3, n)] *= 10.0 ** rng.uniform(-30, -8, n)
    d /= np.abs(d).max(1, keepdims=True)
    both_ways(gpu_ctx, v, np.concatenate([o * size, d], 1).astype(np.float32))


@pytest.mark.gpu
def test_large_and_small_scenes_in_a_batch(gpu_ctx):
    """The scenes of a batch share one unit of the slab distances: the images of each are those of a context of its own."""
    print("[large scenes] batch", flush=True)
    rng = np.random.default_rng(4)
    scenes = [eleven.SceneData.from_arrays(
        (boxes(rng) * size).astype(np.float32).reshape(-1, 9),
        dict(x_res=40, y_res=24, position=(0, 0, -6 * size), focus_distance=float(6 * size)),
        hdri=np.full((2, 4, 3), 0.7, np.float32)) for size in (1.0, 1e12)]
    b = eleven.Batch()
    for k, sc in enumerate(scenes):
        b.add(sc, 4, seed=k)
    b.render(depth=3)
    for k, sc in enumerate(scenes):
        gpu_ctx.upload(sc)
        gpu_ctx.render(4, depth=3, seed=k, rng_scene=k)
        img, n = gpu_ctx.read()[:2]
        rgba, samples = b.read(k)
        assert np.array_equal(samples, n) and np.array_equal(rgba, img) and img[..., :3].max() > 0
    b.close()
