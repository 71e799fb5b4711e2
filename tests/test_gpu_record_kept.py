"""What el_clear does with a record's buffers: up to 2 GiB stay for the next recording render, more goes back."""
import numpy as np
import pytest
import torch

import eleven
from eleven import scenegen


@pytest.mark.gpu
@pytest.mark.parametrize("spp,kept", [(4, True), (24, False)])
def test_large_records_go_back_with_the_accumulation(spp, kept):
    print(f"[record kept] 1024 x 1024 x {spp}, depth 6", flush=True)
    ctx = eleven.Context(0)
    ctx.upload(scenegen.sphere_field_arrays(n_spheres=2, res=(1024, 1024), seed=2))

    def step():
        ctx.clear()
        ctx.render(spp, depth=6, seed=3, flags=eleven.FLAG_RECORD_PATHS)
        return ctx.adjoint(np.ones((1024, 1024, 3), np.float32))[0]
    first = step()
    record = ctx.stats().record_bytes
    assert (record <= 2 << 30) == kept and record >= spp * (1 << 20) * (16 * 7 + 4)
    before = torch.cuda.mem_get_info()[0]
    ctx.clear()
    freed = torch.cuda.mem_get_info()[0] - before
    assert freed == 0 if kept else freed >= record - (64 << 20)
    again = step()
    assert np.linalg.norm(again - first) <= 1e-5 * np.linalg.norm(first)
    ctx.close()
