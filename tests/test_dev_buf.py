"""What a captured launch sequence is compared by (dev_buf.hpp), over a stand-in for the device allocator."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

import eleven
from eleven import scenegen

ROOT = Path(__file__).resolve().parents[1]
HIP = Path("/opt/rocm/include")


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
def test_a_reused_address_is_another_allocation(tmp_path):
    exe = tmp_path / "dev_buf_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{HIP}",
                    f"-I{ROOT / 'tfg-pathtracer_amd' / 'csrc'}", str(ROOT / "tests" / "cpp" / "dev_buf_check.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "bad=0" in r.stdout, r.stdout


@pytest.mark.gpu
def test_a_graph_is_captured_again_after_its_buffers_grew():
    """A captured render, a larger one without a graph, which moves every queue, and the captured one again."""
    print("[graph] buffers grown between two replays", flush=True)
    b = eleven.Batch()
    for i in range(3):
        b.add(scenegen.sphere_field_arrays(n_spheres=4, res=(64, 48), seed=i), 8, seed=i)
    images = {}
    for cap, graph in ((4096, True), (0, False), (4096, True), (0, True), (4096, True)):
        b.render(depth=4, queue_cap=cap, graph=graph)
        images[len(images)] = [b.read(i) for i in range(3)]
    for k in range(1, len(images)):
        for (x, nx), (y, ny) in zip(images[0], images[k]):
            assert np.array_equal(x, y) and np.array_equal(nx, ny)
    assert images[0][0][0][..., :3].max() > 0
    b.close()
