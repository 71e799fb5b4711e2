"""The children that a BVH4 visit leaves on the stack get rows of their own, also where slab distances underflow to zeros
of either sign: the order itself on the host, and hits of directions up to 1e38 long against brute force."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

import eleven
import oracle_py as orc
import raygen
from test_gpu_slabs import QUAD_RAYS, both_ways

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_children_get_rows_of_their_own(tmp_path):
    exe = tmp_path / "child_order_check"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'tfg-pathtracer_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpp" / "child_order_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "bad=0" in r.stdout, r.stdout


def mesh_and_rays(size, length):
    rng = np.random.default_rng(5)
    v = (rng.uniform(-0.5, 0.5, (300, 1, 3)) + rng.normal(scale=0.1, size=(300, 3, 3))).reshape(-1, 9)
    rays = raygen.random_rays(v.astype(np.float32), 2048, seed=7)
    d = rays[:, 3:] / np.linalg.norm(rays[:, 3:], axis=1, keepdims=True)
    o = rng.uniform(-0.6, 0.6, (2048, 3)) - 1.5 * d
    o[:256] = np.round(o[:256] * 8) / 8        # on planes of the grid, and at zero
    return (v * size).astype(np.float32), np.concatenate([o * size, d * length], 1).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("length", [1e33, 1e38])
def test_directions_up_to_1e38(gpu_ctx, length):
    print(f"[child order] directions {length:g} long", flush=True)
    both_ways(gpu_ctx, *mesh_and_rays(1.0, length))


@pytest.mark.gpu
def test_slab_distances_that_are_all_zero(gpu_ctx):
    """A mesh of 1e-10 and directions of 1e38: every slab distance and every t rounds to a zero.  Boxes may be missed
    then (their widening underflows too), but what is found is a hit."""
    print("[child order] all slab distances zero", flush=True)
    v, rays = mesh_and_rays(1e-10, 1e38)
    hit = orc.closest_brute(v, rays)[0] >= 0
    assert 0.1 < hit.mean() < 1
    gpu_ctx.upload(eleven.SceneData.from_arrays(v, camera=dict(x_res=4, y_res=4)))
    reps = QUAD_RAYS // len(rays) + 1
    for r, k in ((rays, 1), (np.tile(rays, (reps, 1)), reps)):
        tri, t, _ = gpu_ctx.trace_closest(r)
        occ = gpu_ctx.trace_any(r, np.full(len(r), np.inf, np.float32))
        found = tri >= 0
        assert (tri < len(v)).all() and not (found & ~np.tile(hit, k)).any() and not (occ & ~np.tile(hit, k)).any()
        assert not t[found].any() and np.isinf(t[~found]).all()
