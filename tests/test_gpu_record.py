"""EL_FLAG_RECORD_PATHS keeps what el_adjoint replays from, and nothing where it has to walk the paths again anyway: plain
renders and wavefront renders deeper than it records."""
import numpy as np
import pytest
import torch

import eleven
from eleven import scenegen


@pytest.mark.gpu
@pytest.mark.parametrize("mode,depth", [(eleven.MODE_PLAIN, 4), (eleven.MODE_WAVEFRONT, 17), (eleven.MODE_PLAIN, 17)])
def test_nothing_is_kept_that_nothing_reads(gpu_ctx, mode, depth):
    print(f"[record] mode {mode}, depth {depth}", flush=True)
    sc = scenegen.sphere_field_arrays(n_spheres=4, res=(256, 192), seed=2)
    gpu_ctx.upload(sc)
    w = np.random.default_rng(1).normal(size=(192, 256, 3)).astype(np.float32)

    def step(flags, m=mode, d=depth):
        gpu_ctx.clear()
        gpu_ctx.render(64, depth=d, seed=3, mode=m, flags=flags)
        return gpu_ctx.read()[:2], gpu_ctx.adjoint(w)[0] if d <= 16 else None
    (im0, n0), g0 = step(0)
    step(eleven.FLAG_RECORD_PATHS, eleven.MODE_WAVEFRONT, 4)
    assert gpu_ctx.stats().record_bytes >= 64 * 192 * 256 * (16 * 4 + 20)
    held = torch.cuda.mem_get_info()[0]
    (im1, n1), g1 = step(eleven.FLAG_RECORD_PATHS)
    assert gpu_ctx.stats().record_bytes == 0
    # the wavefront record's buffers went back
    assert torch.cuda.mem_get_info()[0] >= held + 64 * 192 * 256 * (16 * 4 + 20) - (64 << 20)
    assert np.array_equal(im0, im1) and np.array_equal(n0, n1)
    if g0 is not None:
        # two sums of the same FP32 vertex gradients, in another order of at most 64 FP32 additions before the FP64 sums
        assert np.linalg.norm(g1 - g0) <= 1e-5 * np.linalg.norm(g0)
    with pytest.raises(eleven.ElevenError):
        gpu_ctx.render(1, depth=depth, seed=3, mode=mode, flags=eleven.FLAG_RECORD_PATHS)   # not a cleared accumulation
