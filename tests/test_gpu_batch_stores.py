"""Batched steps whose blocks pass the memory-side cache (column tiles store past it
there) against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

import nebo_hip as nh
from test_gpu_batch_adjoint import _oracle_patch_step

pytestmark = pytest.mark.gpu


def test_column_tiles_of_blocks_past_the_cache():
    dims = [(250, 200, 165), (63, 40, 7), (250, 201, 160)]
    points = [(x + 2) * (y + 2) * (z + 2) for x, y, z in dims]
    assert 16 * sum(points) > 250000000
    coefs = nh.axis_coefs(nh.build_stencils(32, 32, 32, 1.0, 1.0, 1.0))
    s = 0.1 / 32.0 ** 2
    rng = np.random.default_rng(3)
    init = [rng.standard_normal(p) for p in points]
    want = [_oracle_patch_step(d, h, coefs, s) for d, h in zip(dims, init)]
    a, b = nh.alloc_patches(dims)
    for x, h in zip(a, init):
        x.copy_(torch.from_numpy(h))
    for tile in ((0, 1, 4), (0, 2, 8), (0, 4, 16)):
        print(tile, flush=True)
        for x, h in zip(b, init):
            x.copy_(torch.from_numpy(h))
        B = nh.Batch(a, b, dims, coefs, s, tile=tile)
        B.step(swap=0)
        torch.cuda.synchronize()
        for i in range(len(dims)):
            assert np.array_equal(b[i].cpu().numpy(), want[i]), (tile, dims[i])
        B.close()
