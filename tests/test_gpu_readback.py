"""What reaches the caller's arrays: frames and query answers larger than the staging chunk (4 MiB) and on both sides of
its edges, short queries that skip the copies, and accumulations that are emptied by the next render instead of being
cleared."""
import ctypes as C

import numpy as np
import pytest

import eleven
from eleven import scenegen


def passes(ctx, rgba=True, samples=True):
    cam = ctx.camera
    a = np.full((cam.y_res, cam.x_res, 4), 7, np.float32) if rgba else None
    n = np.full((cam.y_res, cam.x_res), 7, np.uint32) if samples else None
    rc = eleven.lib().el_read_passes(ctx._h, a.ctypes.data if rgba else None, n.ctypes.data if samples else None,
                                     C.byref(C.c_uint64()), C.byref(C.c_uint64()))
    assert rc == eleven.EL_OK
    return a, n


@pytest.mark.gpu
@pytest.mark.parametrize("res", [(1, 1), (457, 458), (419430, 1), (209715, 1), (209716, 1), (1920, 1080)])
def test_frames_around_the_chunk(gpu_ctx, res):
    """209,715 pixels of colour and count fill a chunk (262,144 of colour, 1,048,576 of counts): read together and one by
    one, the pieces differ and the values do not."""
    print(f"[readback] {res}", flush=True)
    sc = scenegen.sphere_field_arrays(n_spheres=2, res=res, seed=1)
    gpu_ctx.upload(sc)
    gpu_ctx.render(2, depth=2, seed=3, flags=eleven.FLAG_AOV)
    a, n = passes(gpu_ctx)
    assert n.max() == 2 and np.isfinite(a).all() and (a[..., 3] == 1).all()
    assert np.array_equal(a, passes(gpu_ctx, samples=False)[0])
    assert np.array_equal(n, passes(gpu_ctx, rgba=False)[1])
    nrm = gpu_ctx.read_aov(eleven.PASS_NORMAL)
    assert (nrm[..., 3] == 1).all() and np.abs(nrm[..., :3]).max() <= 1.0001
    rows = np.unique(np.linspace(0, res[0] - 1, 7).astype(int))
    assert a[0, rows].any()


@pytest.mark.gpu
def test_emptied_accumulations(gpu_ctx):
    """clear and set_camera leave the old sums in place until something reads or renders: nothing shows them."""
    print("[readback] clear, set_camera, small generations, plain", flush=True)
    sc = scenegen.sphere_field_arrays(n_spheres=4, res=(40, 24), seed=2)
    gpu_ctx.upload(sc)
    a, n = passes(gpu_ctx)
    assert not a[..., :3].any() and not n.any()
    runs = []
    for mode, cap in ((eleven.MODE_WAVEFRONT, 0), (eleven.MODE_WAVEFRONT, 64), (eleven.MODE_WAVEFRONT, 1536),
                      (eleven.MODE_PLAIN, 0)):
        gpu_ctx.render(3, depth=3, seed=9)   # what must not be seen
        gpu_ctx.clear()
        gpu_ctx.render(2, depth=3, seed=5, mode=mode, queue_cap=cap)
        gpu_ctx.render(1, depth=3, seed=5, mode=mode, queue_cap=cap)
        runs.append(passes(gpu_ctx))
    for a, n in runs[1:3]:
        assert np.array_equal(a, runs[0][0]) and np.array_equal(n, runs[0][1])
    assert np.array_equal(runs[3][1], runs[0][1])
    np.testing.assert_allclose(runs[3][0], runs[0][0], rtol=1e-4, atol=1e-6)
    gpu_ctx.set_camera(sc.camera)
    a, n = passes(gpu_ctx)
    assert not a[..., :3].any() and not n.any()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 262145, 1 << 19])
def test_queries_around_the_direct_size(gpu_ctx, n):
    print(f"[readback] {n} rays", flush=True)
    sc = scenegen.sphere_field_arrays(n_spheres=3, res=(8, 8), seed=4)
    gpu_ctx.upload(sc)
    rng = np.random.default_rng(n)
    o = rng.uniform(-12, 12, (n, 3)) * (1, 0.3, 1)
    d = rng.normal(size=(n, 3))
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    tmax = rng.uniform(0, 20, n).astype(np.float32)
    tri, t, uv = gpu_ctx.trace_closest(rays)
    occ = gpu_ctx.trace_any(rays, tmax)
    assert np.array_equal(occ, (tri >= 0) & (t < tmax))
    for k in {0, n // 2, n - 1}:
        a = max(0, min(k, n - 100))
        one = gpu_ctx.trace_closest(rays[a:a + 100])
        for x, y in zip((tri, t, uv), one):
            assert np.array_equal(x[a:a + 100], y)
    # without the barycentrics
    tri2, t2 = np.zeros(n, np.int32), np.zeros(n, np.float32)
    rc = eleven.lib().el_trace_closest(gpu_ctx._h, rays.ctypes.data, n, tri2.ctypes.data, t2.ctypes.data, None, 0)
    assert rc == eleven.EL_OK and np.array_equal(tri, tri2) and np.array_equal(t, t2)
