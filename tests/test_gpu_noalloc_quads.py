"""el_trace_closest_noalloc at the number of rays up to which a launch goes by quads, which need none of its spill area,
and beyond, where the area bounds the threads: both find what el_trace_closest finds."""
import numpy as np
import pytest

import eleven
import raygen
from eleven import scenegen
from test_gpu_slabs import QUAD_RAYS


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, QUAD_RAYS, QUAD_RAYS + 1])
def test_noalloc_on_both_sides_of_the_quads(gpu_ctx, scene_root, n):
    print(f"[no-alloc] {n} rays", flush=True)
    scene = eleven.SceneData.load(scenegen.heightfield(scene_root / "noalloc_quads", cells=(256, 128), extent=(25.6, 12.8),
                                                       res=(96, 54), n_mats=4, tex_size=16, sky=(32, 16)))
    gpu_ctx.upload(scene)
    rays = raygen.random_rays(scene.vertices(), n, seed=9)
    tri, t, uv = gpu_ctx.trace_closest(rays)
    dr, dtri, dt, duv = (gpu_ctx.alloc(b) for b in (rays.nbytes, 4 * n, 4 * n, 8 * n))
    try:
        gpu_ctx.htod(dr, rays)
        gpu_ctx.trace_closest_noalloc(dr, n, dtri, dt, duv)
        for want, src in ((tri, dtri), (t, dt), (uv, duv)):
            got = np.empty_like(want)
            gpu_ctx.dtoh(got, src)
            assert np.array_equal(got, want)
    finally:
        for p in (dr, dtri, dt, duv):
            gpu_ctx.free(p)
