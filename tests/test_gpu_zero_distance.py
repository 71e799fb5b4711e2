"""Rays that start on the mesh: every triangle around their origin is hit at a distance of 0 or -0, and the lowest index of
them is the closest hit.  A closest hit at -0 leaves no part of the tree out."""
import numpy as np
import pytest

import eleven
import oracle_py as orc
from test_gpu_slabs import QUAD_RAYS


@pytest.mark.gpu
@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_lowest_index_of_the_hits_at_zero(gpu_ctx, axis, width):
    print(f"[zero distance] plane across axis {axis}, BVH{width}", flush=True)
    rng = np.random.default_rng(axis)
    n = 24
    i, j = np.meshgrid(np.arange(n), np.arange(n))
    i, j = i.ravel(), j.ravel()
    corner = lambda a, b: np.stack([np.zeros_like(a), a, b], -1)  # noqa: E731
    f = np.concatenate([np.stack([corner(i, j), corner(i + 1, j), corner(i + 1, j + 1)], 1),
                        np.stack([corner(i, j), corner(i + 1, j + 1), corner(i, j + 1)], 1)]).astype(np.float32)
    f[::2] = f[::2, [0, 2, 1]]                      # both windings: determinants, and zeros, of either sign
    f = np.roll(f[rng.permutation(len(f))], axis, axis=2)   # the indices of neighbours far apart
    v = np.ascontiguousarray(f).reshape(-1, 9)
    m = 4096
    o = np.roll(np.concatenate([np.zeros((m, 1)), rng.integers(0, 2 * n + 1, (m, 2)) / 2], 1), axis, axis=1)
    d = rng.normal(size=(m, 3))
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    tb, tt, _, _ = orc.closest_brute(v, rays)
    assert (tb >= 0).mean() > 0.9 and np.signbit(tt[tb >= 0]).any() and not tt[tb >= 0].any()
    gpu_ctx.upload(eleven.SceneData.from_arrays(v, camera=dict(x_res=8, y_res=8)))
    gpu_ctx.render(1, depth=1, bvh_width=width)
    reps = QUAD_RAYS // m + 1
    for r, k in ((rays, 1), (np.tile(rays, (reps, 1)), reps)):   # by quads, and by lanes
        tri, t, _ = gpu_ctx.trace_closest(r)
        assert np.array_equal(tri, np.tile(tb, k)) and np.array_equal(t, np.tile(tt, k))
    gpu_ctx.render(1, depth=1, bvh_width=4)
