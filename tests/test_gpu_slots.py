"""Generations of whole frames keep the samples of a tile together, all others go frame after frame: the same image, bit
for bit, however a render or a batch is cut into generations (runs of 1, 2, 3, 7 and all samples, and parts of a
frame), at sizes with ragged tiles."""
import numpy as np
import pytest

import eleven
from eleven import scenegen

SPP = 7


def tiles(w, h):
    return (w + 7) // 8 * ((h + 7) // 8) * 64


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(8, 8), (1, 1), (13, 9), (40, 24)])
def test_generations_of_a_render(gpu_ctx, w, h):
    print(f"[slots] {w}x{h}", flush=True)
    gpu_ctx.upload(scenegen.sphere_field_arrays(n_spheres=6, res=(w, h), seed=3))
    n = tiles(w, h)
    want = None
    for cap in (64, 0, n, 2 * n, 3 * n, n + 64, SPP * n):
        gpu_ctx.clear()
        gpu_ctx.render(2, depth=4, seed=9, queue_cap=cap)
        gpu_ctx.render(SPP, depth=4, seed=9, queue_cap=cap)
        got = gpu_ctx.read()
        want = want or got
        for x, y in zip(got[:2], want[:2]):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), cap
        assert got[2:] == want[2:]
    assert want[1].max() > 0   # a pixel's NaN samples are not counted


@pytest.mark.gpu
def test_generations_of_a_batch():
    print("[slots] batch", flush=True)
    sizes = [(13, 9), (40, 24), (8, 8), (17, 16)]
    scenes = [scenegen.sphere_field_arrays(n_spheres=4, res=s, seed=i) for i, s in enumerate(sizes)]
    total = SPP * sum(tiles(*s) for s in sizes)
    want = None
    b = eleven.Batch(0)
    for i, s in enumerate(scenes):
        b.add(s, SPP, i + 3)
    for cap in (64, 0, 256, 1536, 5 * 960, total):
        b.render(depth=4, queue_cap=cap)
        got = [b.read(i) for i in range(4)]
        want = want or got
        for x, y in zip(got, want):
            assert all(np.array_equal(p, q) for p, q in zip(x, y)), cap
    b.close()
