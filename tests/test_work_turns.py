"""How a launch's chunks go to its waves in turn, on the host (work_turns.hpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_chunk_once_and_none_after_the_last(tmp_path):
    exe = tmp_path / "work_turns_check"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'tfg-pathtracer_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpp" / "work_turns_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "bad=0" in r.stdout, r.stdout
