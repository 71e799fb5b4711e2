"""Device memory of an adjoint: the plan on the host (adjoint_plan.hpp), and what a first adjoint at the largest depth takes."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch

import eleven
from eleven import scenegen

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_generations_within_their_memory(tmp_path):
    exe = tmp_path / "adjoint_plan_check"
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{ROOT / 'tfg-pathtracer_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpp" / "adjoint_plan_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "bad=0" in r.stdout, r.stdout


@pytest.mark.gpu
def test_an_adjoint_takes_two_gibibytes_at_most():
    """512 x 512 x 16 paths of depth 16, after a plain render: no queues are there yet."""
    print("[adjoint memory] depth 16", flush=True)
    ctx = eleven.Context(0)
    ctx.upload(scenegen.sphere_field_arrays(n_spheres=4, res=(512, 512), seed=1))
    ctx.render(16, depth=16, seed=1, mode=eleven.MODE_PLAIN)
    w = np.ones((512, 512, 3), np.float32)
    before = torch.cuda.mem_get_info()[0]
    grad, _ = ctx.adjoint(w)
    # beside the generation: the image and the sums, and what the allocator rounds up (2 MiB a buffer)
    assert before - torch.cuda.mem_get_info()[0] <= (2 << 30) + w.nbytes + 18 * (2 << 20)
    assert np.isfinite(grad).all() and np.abs(grad).max() > 0
    ctx.close()
