"""nebo_last_backend names the store policy a stencil tile runs with: the one-wave tiles
write back as Euler steps and store past the caches as assignments."""
import pytest
import torch

import nebo_hip as nh
from nebo_hip import adjoint as adj

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,step,assignment", [((64, 2, 8, 3), True, False), ((128, 8, 64, 7), False, False),
                                                  ((128, 8, 64, 9), True, True), ((128, 8, 64, 11), False, False)])
def test_store_policy(tile, step, assignment):
    n = (128, 16, 64)
    L = nh.Layout.build(n, 1)
    c = nh.axis_coefs(nh.build_stencils(*n, 1.0, 1.0, 1.0))
    k, phi, out = (nh.Field.from_numpy(L, torch.rand(L.npts, dtype=torch.float64).numpy(), where="gpu")
                   for _ in range(3))
    nh.stencil_set_tile(0, *tile)
    try:
        nh.divkgrad(out, k, phi, c)
        assert ("write-back" in nh.last_backend()) == assignment, nh.last_backend()
        adj.diffusion_step(L, out.gpu, phi.gpu, k.gpu, c, 1e-4)
        assert ("write-back" in nh.last_backend()) == step, nh.last_backend()
    finally:
        nh.stencil_reset_tile(0)
    torch.cuda.synchronize()
