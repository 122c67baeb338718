"""The tile rule of the hand-written stencil kernels on boxes whose sides suit no
tile: what it picks on a GPU of 256 compute units (the fallback where there is none),
and that the pick gives the oracle's bits."""
import numpy as np
import pytest

import nebo_hip as nh

BIG, DEF, PAIR = (64, 4, 8, 3), (128, 8, 64, 7), (128, 8, 64, 11)
RULE = [
    # box, div(k grad phi), Laplacian + Euler
    ((224, 224, 224), DEF, DEF),                    # 0.67 of the CUs' cells
    ((300, 210, 170), BIG, BIG),                    # 0.64
    ((256, 128, 256), BIG, (64, 2, 8, 3)),          # half the CUs
    ((256, 256, 250), PAIR, DEF),
    ((300, 300, 300), BIG, BIG),                    # past the 128-plane chunks
    ((512, 512, 100), (128, 8, 512, 7), (128, 8, 512, 7)),
    ((200, 190, 210), BIG, (64, 2, 8, 3)),
    ((160, 160, 160), (64, 2, 8, 3), (64, 2, 8, 3)),
    ((180, 150, 130), (64, 2, 16, 3), (64, 2, 16, 3)),
    ((100, 100, 100), (64, 2, 8, 3), (64, 2, 8, 3)),
    ((90, 70, 80), (64, 2, 4, 3), (64, 2, 4, 3)),
    ((1, 1, 1), (64, 2, 4, 3), (64, 2, 4, 3)),
]


@pytest.mark.parametrize("box,divk,lapl", RULE)
def test_tile_of_a_box(box, divk, lapl):
    assert nh.stencil_select_tile(0, box) == divk
    assert nh.stencil_select_tile(1, box) == lapl


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(131, 50, 90), (300, 90, 110), (66, 130, 200)])
def test_ragged_boxes_bit_exact(n):
    import torch
    import oracle_lib as orc
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(sum(n))
    k, phi = (nh.Field.from_numpy(L, rng.uniform(0.5, 2.0, L.npts)) for _ in range(2))
    c = nh.axis_coefs(nh.build_stencils(*n, 1.0, 1.0, 1.0))
    for run, want in ((nh.divkgrad, orc.divkgrad), (nh.lapl_euler, orc.lapl_euler)):
        r, ref = (nh.Field.from_numpy(L, np.zeros(L.npts), where=w) for w in ("gpu", "cpu"))
        args = (k, phi, c) if run is nh.divkgrad else (phi, c, 0.01)
        run(r, *args)
        want(ref, *args, *((0,) if run is nh.divkgrad else ()))
        torch.cuda.synchronize()
        assert np.array_equal(r.gpu.cpu().numpy(), ref.host), run
