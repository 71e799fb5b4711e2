"""Gradients come back the same on both sides of the sizes at which their copies change course: textures and material
tables of 1 MiB (a texel is 12 bytes, a material 48)."""
import numpy as np
import pytest

import eleven
from test_gpu_adjoint_replay import close, grads, plane_scene


@pytest.mark.gpu
@pytest.mark.parametrize("size", [295, 296])
def test_texel_gradients_of_one_mebibyte(gpu_ctx, size):
    """The texel gradients of a constant texture sum to the gradient of a scalar albedo of its value."""
    print(f"[adjoint results] {size} x {size} texels", flush=True)
    tex = np.full((size, size, 3), 0.4, np.float32)
    sc = plane_scene((160, 90), tex, 1)
    gpu_ctx.upload(sc)
    dmat, dtex = grads(gpu_ctx, sc, 8, 3)
    again, tagain = gpu_ctx.adjoint(np.zeros((90, 160, 3), np.float32), grad_texture=0, accumulate=True)
    assert np.array_equal(again, dmat) and np.array_equal(tagain, dtex)   # nothing was added: the same sums
    plain = plane_scene((160, 90), tex, 1, materials=2, used=1)
    mats = plain.materials()
    mats[1].albedo_tex = -1
    mats[1].albedo = eleven.float3(0.4, 0.4, 0.4)
    gpu_ctx.upload(plain)
    want, _ = grads(gpu_ctx, plain, 8, 3, tex=-1)
    # texel sums are FP32 atomics of up to a few thousand terms a texel
    assert close(dtex.sum(axis=(0, 1), dtype=np.float64), want[1, :3], 1e-4) and want[1, :3].all()


@pytest.mark.gpu
@pytest.mark.parametrize("materials", [21845, 21846])
def test_material_gradients_of_one_mebibyte(gpu_ctx, materials):
    print(f"[adjoint results] {materials} materials", flush=True)
    tex = np.random.default_rng(2).uniform(0.1, 0.9, (8, 8, 3)).astype(np.float32)
    one_scene = plane_scene((64, 48), tex, 0)
    gpu_ctx.upload(one_scene)
    one, tone = grads(gpu_ctx, one_scene, 8, 3)
    sc = plane_scene((64, 48), tex, 0, materials, materials - 1)
    gpu_ctx.upload(sc)
    many, tmany = grads(gpu_ctx, sc, 8, 3)
    # sums of the same FP32 vertex gradients: at most 64 FP32 additions before the FP64 ones, and FP32 atomics
    assert close(many[-1], one[0], 1e-5) and not many[:-1].any() and one.any() and close(tmany, tone, 1e-4)
