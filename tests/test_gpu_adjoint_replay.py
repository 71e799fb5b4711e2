"""The bounce-by-bounce path replay of el_adjoint at the sizes where it changes course: more paths than one generation
holds, more materials than the LDS sums hold, frames of a few pixels, and texel gradients of magnified textures (summed
in the wave) and minified ones (every lane by itself).

The vertex gradients of the compared runs are the same FP32 values; only the order of their sums differs, at most 64
FP32 additions before the FP64 (material) sums: 1e-5 of the gradient's norm covers 64 x 2^-24 = 4e-6.  Texel sums are
FP32 atomics of up to a few thousand terms a texel: 1e-4."""
import numpy as np
import pytest

import eleven
from eleven import make_material, make_texture, scenegen


def grads(ctx, sc, spp, depth, flags=0, weight=None, tex=0):
    H, W = sc.camera.y_res, sc.camera.x_res
    w = np.random.default_rng(3).normal(size=(H, W, 3)).astype(np.float32) if weight is None else weight
    ctx.clear()
    ctx.render(spp, depth=depth, seed=11, flags=flags)
    return ctx.adjoint(w, grad_texture=tex)


def close(a, b, tol):
    return np.linalg.norm(a.astype(np.float64) - b) <= tol * np.linalg.norm(b.astype(np.float64))


def plane_scene(res, texture, filt, materials=1, used=0):
    """A textured ground plane under a sky, seen from above."""
    v = np.array([[-20, 0, -20, 20, 0, -20, 20, 0, 20], [-20, 0, -20, 20, 0, 20, -20, 0, 20]], np.float32)
    uv = np.array([[0, 0, 1, 0, 1, 1], [0, 0, 1, 1, 0, 1]], np.float32)
    mats = [make_material(albedo=(0.5, 0.4, 0.3), roughness=0.7, albedo_tex=0 if i == used else -1)
            for i in range(materials)]
    return eleven.SceneData.from_arrays(
        v, dict(x_res=res[0], y_res=res[1], position=(0, 8, -25), rotation=(17.7, 0, 0)),
        normals=np.tile([0.0, 1.0, 0.0], (2, 3)).reshape(2, 9), uvs=uv, object_id=np.zeros(2, np.int32),
        mesh_material=np.array([used]), materials=mats, textures=[make_texture(texture, filt=filt)],
        hdri=scenegen.sky_hdr(64, 32, peak=20.0, sigma_deg=10.0), lights=[((2, 6, 0), (30, 30, 30))])


@pytest.mark.gpu
@pytest.mark.parametrize("res,spp,depth", [((1, 1), 1, 1), ((13, 7), 3, 16), ((512, 512), 40, 6)])
def test_traced_equals_recorded(gpu_ctx, res, spp, depth):
    """512 x 512 x 40 paths are more than one generation of the traced walk and of the recorded replay."""
    print(f"[replay] {res} {spp} spp depth {depth}", flush=True)
    sc = plane_scene(res, np.random.default_rng(1).uniform(0.1, 0.9, (8, 8, 3)).astype(np.float32), 1)
    gpu_ctx.upload(sc)
    m1, t1 = grads(gpu_ctx, sc, spp, depth)
    m2, t2 = grads(gpu_ctx, sc, spp, depth, flags=eleven.FLAG_RECORD_PATHS)
    assert gpu_ctx.stats().adjoint_rays == 0
    assert close(m1, m2, 1e-5) and close(t1, t2, 1e-4)
    if res != (1, 1):
        assert np.abs(m2).max() > 0 and np.abs(t2).max() > 0


@pytest.mark.gpu
@pytest.mark.parametrize("materials", [512, 513, 1000])
def test_many_materials_equal_one(gpu_ctx, materials):
    print(f"[replay] {materials} materials", flush=True)
    tex = np.random.default_rng(2).uniform(0.1, 0.9, (8, 8, 3)).astype(np.float32)
    gpu_ctx.upload(plane_scene((64, 48), tex, 0))
    one, _ = grads(gpu_ctx, plane_scene((64, 48), tex, 0), 8, 3)
    sc = plane_scene((64, 48), tex, 0, materials, materials - 1)
    gpu_ctx.upload(sc)
    many, _ = grads(gpu_ctx, sc, 8, 3)
    assert close(many[-1], one[0], 1e-5) and not many[:-1].any() and one.any()


@pytest.mark.gpu
@pytest.mark.parametrize("filt", [0, 1])
@pytest.mark.parametrize("size", [1, 2, 16, 700])
def test_texel_gradients_sum_to_the_albedo_gradient(gpu_ctx, filt, size):
    """The bilinear weights of a vertex sum to 1 and an untextured albedo has the gradient that the texels share, so the
    texel gradients of a constant texture sum to the gradient of a scalar albedo of that value, whether lanes are
    summed in the wave (1 to 16 texels across the plane) or not (700)."""
    print(f"[replay] {size} x {size} texels, filter {filt}", flush=True)
    tex = np.full((size, size, 3), 0.4, np.float32)
    sc = plane_scene((160, 90), tex, filt)
    gpu_ctx.upload(sc)
    _, dtex = grads(gpu_ctx, sc, 8, 3)
    plain = plane_scene((160, 90), tex, filt, materials=2, used=1)
    mats = plain.materials()
    mats[1].albedo_tex = -1
    mats[1].albedo = eleven.float3(0.4, 0.4, 0.4)
    gpu_ctx.upload(plain)
    dmat, _ = grads(gpu_ctx, plain, 8, 3, tex=-1)
    assert close(dtex.sum(axis=(0, 1), dtype=np.float64), dmat[1, :3], 1e-4) and dmat[1, :3].all()
