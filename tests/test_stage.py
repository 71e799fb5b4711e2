"""The pinned memory between the GPU and callers' arrays (stage.hpp): on the host over a stand-in for the runtime, and
contexts and a batch's scenes read by several threads at once."""
import shutil
import subprocess
import threading
from pathlib import Path

import numpy as np
import pytest

import eleven
from eleven import scenegen

ROOT = Path(__file__).resolve().parents[1]
HIP = Path("/opt/rocm/include")


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
@pytest.mark.parametrize("mode", ["pool", "copy"])
def test_stages_on_the_host(tmp_path, mode):
    exe = tmp_path / "stage_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{HIP}",
                    f"-I{ROOT / 'tfg-pathtracer_amd' / 'csrc'}", str(ROOT / "tests" / "cpp" / "stage_check.cpp"),
                    "-o", str(exe), "-lpthread"], check=True)
    r = subprocess.run([str(exe), mode], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "bad=0" in r.stdout, r.stdout


def in_threads(n, f):
    got, errors = [None] * n, []

    def go(i):
        try:
            got[i] = f(i)
        except Exception as e:  # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=go, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    return got


@pytest.mark.gpu
def test_scenes_of_a_batch_read_by_several_threads():
    print("[stage] four threads read a batch", flush=True)
    b = eleven.Batch()
    sizes = [(320, 200), (64, 48), (500, 333), (17, 9)]
    for i, res in enumerate(sizes):
        b.add(scenegen.sphere_field_arrays(n_spheres=3, res=res, seed=i), 2, seed=i)
    b.render(depth=3)
    alone = [b.read(i) for i in range(4)]
    for _ in range(5):
        for (x, nx), (y, ny) in zip(alone, in_threads(4, b.read)):
            assert np.array_equal(x, y) and np.array_equal(nx, ny)
    b.close()


@pytest.mark.gpu
def test_contexts_in_several_threads():
    print("[stage] four contexts in four threads", flush=True)

    def step(i):
        out = []
        c = eleven.Context(0)
        sc = scenegen.sphere_field_arrays(n_spheres=4, res=(200 + 70 * i, 150), seed=i)
        c.upload(sc)
        rays = np.random.default_rng(i).normal(size=(500 + 9000 * i, 6)).astype(np.float32)
        for k in range(3):
            c.clear()
            c.render(2, depth=3, seed=i)
            out += [*c.read()[:2], *c.trace_closest(rays), *c.adjoint(np.ones((150, 200 + 70 * i, 3), np.float32))[:1]]
        c.close()
        return out
    alone = [step(i) for i in range(4)]
    for x, y in zip(alone, in_threads(4, step)):
        for k, (a, b) in enumerate(zip(x, y)):
            # the material gradients (every sixth) are sums of atomics
            assert np.allclose(a, b, rtol=1e-5, atol=1e-6) if k % 6 == 5 else np.array_equal(a, b)


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
def test_helpers_sleep_while_the_gpu_works(tmp_path):
    test_stages_on_the_host(tmp_path, "wait")


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
def test_a_stage_for_each_context(tmp_path):
    test_stages_on_the_host(tmp_path, "contexts")
