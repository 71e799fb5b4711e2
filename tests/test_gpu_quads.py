"""Short launches trace a ray with four lanes, long ones (more than 2^20 rays) with one: both find the closest hit of
the brute-force oracle and of each other, bit for bit, at the sizes where a wave's 16 rays run out, on a tree deeper
than the quads' stack, and for directions with zero, infinite and NaN components."""
import numpy as np
import pytest

import eleven
import oracle_py as orc
import raygen
from eleven import scenegen

QUAD_RAYS = 1 << 20


@pytest.fixture(scope="module")
def field():
    return scenegen.sphere_field_arrays(n_spheres=6, res=(16, 16), seed=3)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 63, 64, 65, 1000, 8192])
def test_short_launches_equal_brute_force(gpu_ctx, field, n):
    print(f"[quads] {n} rays", flush=True)
    gpu_ctx.upload(field)
    v = field.vertices()
    rays = raygen.random_rays(v, n, seed=n)
    tri, t, uv = gpu_ctx.trace_closest(rays)
    tb, tt, ub, vb = orc.closest_brute(v, rays)
    hit = tb >= 0
    assert np.array_equal(tri, tb) and np.array_equal(t[hit], tt[hit]) and np.isinf(t[~hit]).all()
    assert np.array_equal(uv[hit, 0], ub[hit]) and np.array_equal(uv[hit, 1], vb[hit])
    tmax = np.random.default_rng(n).uniform(0, 30, n).astype(np.float32)
    assert np.array_equal(gpu_ctx.trace_any(rays, tmax), hit & (t < tmax))


@pytest.mark.gpu
@pytest.mark.parametrize("scene", ["field", "soup"])
def test_quads_equal_lanes(gpu_ctx, field, scene):
    print(f"[quads] {scene}: one long launch against short ones", flush=True)
    rng = np.random.default_rng(8)
    if scene == "soup":   # leaves of up to 8 triangles, every third triangle twice
        v = (rng.uniform(-1, 1, (3000, 1, 3)) + rng.normal(scale=0.05, size=(3000, 3, 3))).astype(np.float32)
        v[1::3] = v[::3]
        field = eleven.SceneData.from_arrays(v.reshape(-1, 9), camera=dict(x_res=4, y_res=4))
    gpu_ctx.upload(field)
    n = QUAD_RAYS + 3
    rays = raygen.random_rays(field.vertices(), n, seed=5)
    odd = rays[:64, 3:]
    odd[:16, 0] = odd[16:32, 1] = odd[24:48, 2] = 0.0
    odd[48:52, 1] = np.inf
    odd[52:56, 2] = np.nan
    odd[56:] = 0.0
    tmax = rng.uniform(0, 4, n).astype(np.float32)
    tmax[100:104] = np.inf, np.nan, 0.0, -1.0
    long = gpu_ctx.trace_closest(rays) + (gpu_ctx.trace_any(rays, tmax),)
    cuts = [0, 7, 16, 1024, 200000, QUAD_RAYS, n]
    for a, b in zip(cuts, cuts[1:]):
        short = gpu_ctx.trace_closest(rays[a:b]) + (gpu_ctx.trace_any(rays[a:b], tmax[a:b]),)
        for x, y in zip(long, short):
            assert np.array_equal(x[a:b], y, equal_nan=True), (a, b)


@pytest.mark.gpu
def test_tree_deeper_than_the_quads_stack(gpu_ctx):
    print("[quads] a chain of triangles, each a tenth larger and farther", flush=True)
    x = 1e-6 * 1.1 ** np.arange(360)
    s = 0.2 * x
    z = np.zeros_like(x)
    v = np.stack([x, z, z, x + s, s, z, x, s, s], -1).astype(np.float32)
    sc = eleven.SceneData.from_arrays(v, camera=dict(x_res=32, y_res=32), lights=[((0, 5, 0), (1, 1, 1))])
    gpu_ctx.upload(sc)
    assert gpu_ctx.stats().stack_bound > 62   # stays on the lanes' path, whose stack spills
    rng = np.random.default_rng(1)
    pick = rng.integers(0, len(v), 4000)
    target = v.reshape(-1, 3, 3)[pick].mean(1)
    o = (target + rng.normal(size=target.shape) * np.abs(target[:, :1])).astype(np.float32)
    d = target - o
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    tri, t, _ = gpu_ctx.trace_closest(rays)
    tb, tt, _, _ = orc.closest_brute(v, rays)
    assert np.array_equal(tri, tb) and np.array_equal(t[tb >= 0], tt[tb >= 0]) and (tb >= 0).any()
    assert gpu_ctx.render(2, depth=3, seed=1).paths == 2 * 32 * 32


@pytest.mark.gpu
@pytest.mark.parametrize("side,spp,width", [(8, 1, 4), (9, 3, 4), (40, 5, 8), (200, 9, 4), (512, 6, 4), (512, 2, 8)])
def test_queues_in_one_launch_equal_launches_of_their_own(gpu_ctx, side, spp, width):
    """A bounce's shadow queues and the next closest hits in one launch, its waves divided among them (a wave a chunk,
    or in proportion to the rays), against a launch for each."""
    print(f"[quads] {side}x{side} {spp} spp width {width}", flush=True)
    gpu_ctx.upload(scenegen.sphere_field_arrays(n_spheres=20, res=(side, side), seed=2))
    out = []
    for flags in (0, eleven.FLAG_SERIAL_SHADOWS, 0):
        gpu_ctx.clear()
        st = gpu_ctx.render(spp, depth=5, seed=4, bvh_width=width, flags=flags)
        img, cnt, rays, verts = gpu_ctx.read()
        out.append((img.view(np.uint32), cnt, rays, verts, st.extend_rays))
    gpu_ctx.render(1, depth=1, bvh_width=4)   # the context is shared: back to the default tree
    for o in out[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(out[0], o))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [131072, 131073, 262144 - 15, 262144 + 16, 393216 + 1, 917504, (1 << 22) + 65, 10_000_001])
def test_every_chunk_is_traced_once(gpu_ctx, field, n):
    """Full and partial turns of a launch's waves (8,192 x 16 rays a turn by quads, 8,192 x 64 and more by lanes): every
    ray is answered as in a launch of its own part."""
    print(f"[quads] {n} rays in turns", flush=True)
    gpu_ctx.upload(field)
    some = raygen.random_rays(field.vertices(), 1 << 16, seed=21)
    want = gpu_ctx.trace_closest(some)
    rays = np.tile(some, ((n + len(some) - 1) // len(some), 1))[:n]
    got = gpu_ctx.trace_closest(rays)
    for x, y in zip(got, want):
        assert np.array_equal(x, np.concatenate([y] * ((n + len(y) - 1) // len(y)))[:n])
    occ = gpu_ctx.trace_any(rays, np.full(n, np.inf, np.float32))
    assert np.array_equal(occ, got[0] >= 0)
