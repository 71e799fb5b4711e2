"""Ray queries on both sides of the number of rays up to which they go by quads of lanes."""
import numpy as np
import pytest

import eleven
import oracle_py as orc
import raygen

QUERY_QUAD_RAYS = 3 << 17


@pytest.mark.gpu
@pytest.mark.parametrize("n", [QUERY_QUAD_RAYS - 1, QUERY_QUAD_RAYS, QUERY_QUAD_RAYS + 1])
def test_queries_on_both_sides_of_the_line(gpu_ctx, n):
    print(f"[query line] {n} rays", flush=True)
    rng = np.random.default_rng(8)
    v = (rng.uniform(-1, 1, (300, 1, 3)) + rng.normal(scale=0.2, size=(300, 3, 3))).astype(np.float32).reshape(-1, 9)
    rays = raygen.random_rays(v, 2048, seed=3)
    tb, tt, _, _ = orc.closest_brute(v, rays)
    far = np.where(rng.random(2048) < 0.5, np.inf, rng.uniform(0, 2, 2048)).astype(np.float32)
    idx = np.arange(n) % 2048
    gpu_ctx.upload(eleven.SceneData.from_arrays(v, camera=dict(x_res=4, y_res=4)))
    tri, t, _ = gpu_ctx.trace_closest(rays[idx])
    hit = tb >= 0
    assert np.array_equal(tri, tb[idx]) and np.array_equal(t[hit[idx]], tt[idx][hit[idx]])
    occ = gpu_ctx.trace_any(rays[idx], far[idx])
    assert np.array_equal(occ, (hit & (tt < far))[idx])
