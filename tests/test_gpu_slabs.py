"""The slab tests of the traversal never lose a hit that brute force finds: directions from 1e-9 to 1e20 long (slab
distances are kept in another unit from 2^20 on), with components down to zero, and nodes so small and far away that
the inverted boxes of their empty slots pass the test.  Both by quads and, more than 2^20 rays, by lanes."""
import numpy as np
import pytest

import eleven
import oracle_py as orc
import raygen

QUAD_RAYS = 1 << 20


def both_ways(ctx, v, rays):
    ctx.upload(eleven.SceneData.from_arrays(v, camera=dict(x_res=4, y_res=4)))
    tb, tt, _, _ = orc.closest_brute(v, rays)
    hit = tb >= 0
    assert hit.any()
    reps = QUAD_RAYS // len(rays) + 1
    for r, k in ((rays, 1), (np.tile(rays, (reps, 1)), reps)):
        tri, t, _ = ctx.trace_closest(r)
        occ = ctx.trace_any(r, np.full(len(r), np.inf, np.float32))
        assert np.array_equal(tri, np.tile(tb, k)) and np.array_equal(occ, np.tile(hit, k))
        assert np.array_equal(t[np.tile(hit, k)], np.tile(tt[hit], k))


@pytest.mark.gpu
@pytest.mark.parametrize("length", [1e-9, 1e-3, 1.0, 2.0**20, 2.0**20 * 1.01, 1e12, 1e20])
def test_directions_of_any_length(gpu_ctx, length):
    print(f"[slabs] directions {length:g} long", flush=True)
    rng = np.random.default_rng(4)
    v = (rng.uniform(-500, 500, (400, 1, 3)) + rng.normal(scale=60, size=(400, 3, 3))).astype(np.float32).reshape(-1, 9)
    rays = raygen.random_rays(v, 2048, seed=6)
    rays[:64, 3] = 0.0
    rays[32:96, 4] *= np.float32(1e-27)
    rays[96:128, 3:5] = -0.0
    rays[:, 3:] *= np.float32(length)
    both_ways(gpu_ctx, v, rays)


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 2, 3, 5, 9, 33])
def test_nodes_below_the_rounding_of_their_distance(gpu_ctx, count):
    print(f"[slabs] {count} triangles of 0.001 at 2000", flush=True)
    rng = np.random.default_rng(count)
    c = np.float32([2000, -1500, 1800]) + rng.uniform(0, 0.002, (count, 1, 3))
    v = (c + rng.normal(scale=0.001, size=(count, 3, 3))).astype(np.float32).reshape(-1, 9)
    o = rng.uniform(-1, 1, (1024, 3)).astype(np.float32)
    d = v.reshape(-1, 3, 3)[rng.integers(0, count, 1024)].mean(1) - o
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    rays[::3, 3:] *= 1000   # the determinant's threshold is absolute
    both_ways(gpu_ctx, v, rays)
