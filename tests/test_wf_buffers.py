"""The wavefront buffers when the device runs out of memory (wf_buffers.hpp), over a stand-in for its allocator."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIP = Path("/opt/rocm/include")


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
def test_a_failed_growth_leaves_every_buffer_usable(tmp_path):
    exe = tmp_path / "wf_buffers_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{HIP}",
                    f"-I{ROOT / 'tfg-pathtracer_amd' / 'csrc'}", str(ROOT / "tests" / "cpp" / "wf_buffers_check.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "bad=0" in r.stdout, r.stdout
