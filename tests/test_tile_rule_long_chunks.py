"""The long-chunk tile of the hand-written stencil kernels: boxes it divides whose rounds
of workgroups are nearly empty leave it, boxes it does not divide whose rounds are
full take it, and its last chunk's bits."""
import numpy as np
import pytest

import nebo_hip as nh

BIG, DEF, PAIR = (64, 4, 8, 3), (128, 8, 64, 7), (128, 8, 64, 11)
LONG = {z: (128, 8, z, 7) for z in (128, 256, 512)}
RULE = [
    # box, div(k grad phi), Laplacian + Euler
    ((512, 512, 512), LONG[512], LONG[512]),
    ((512, 256, 512), LONG[256], LONG[256]),
    ((256, 512, 200), LONG[128], LONG[128]),        # one round of 256 workgroups, 0.78
    ((512, 512, 40), LONG[512], LONG[512]),
    ((500, 512, 100), LONG[512], LONG[512]),        # not divided; one round
    ((500, 512, 30), LONG[512], LONG[512]),         # not divided, and thin
    ((1000, 1000, 9), BIG, BIG),                    # too thin
    ((1500, 700, 10), LONG[512], LONG[512]),
    ((2048, 2048, 4), BIG, BIG),
    ((256, 400, 300), PAIR, DEF),                   # 300 workgroups of 128 planes: 0.46
    ((384, 512, 200), PAIR, DEF),                   # 384: 0.59
    ((512, 384, 512), PAIR, DEF),                   # 384 of 256 planes: 0.75
    ((640, 640, 640), PAIR, DEF),                   # 800 of 512 planes: 0.49
    ((896, 256, 130), BIG, BIG),                    # and the default tile's are as empty
]


@pytest.mark.parametrize("box,divk,lapl", RULE)
def test_tile_of_a_box(box, divk, lapl):
    assert nh.stencil_select_tile(0, box) == divk
    assert nh.stencil_select_tile(1, box) == lapl


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(500, 512, 65), (384, 512, 90)])
def test_bits_of_both_sides_of_the_line(n):
    import torch
    import oracle_lib as orc
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(sum(n))
    k, phi = (nh.Field.from_numpy(L, rng.uniform(0.5, 2.0, L.npts)) for _ in range(2))
    c = nh.axis_coefs(nh.build_stencils(*n, 1.0, 1.0, 1.0))
    r, ref = (nh.Field.from_numpy(L, np.zeros(L.npts), where=w) for w in ("gpu", "cpu"))
    nh.divkgrad(r, k, phi, c)
    orc.divkgrad(ref, k, phi, c, 0)
    torch.cuda.synchronize()
    assert np.array_equal(r.gpu.cpu().numpy(), ref.host)
