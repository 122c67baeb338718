"""The schedule of transport stages by box: the 128 x 8 tile by the planes its rounds of
workgroups walk, on a GPU of 256 compute units (the fallback where there is none), and
the bits on both sides of that line against the direct schedule's."""
import pytest

import nebo_hip as nh
from nebo_hip import transport as tr

TILE, DIRECT, WAVE = tr.SCHED_COLUMN_PF1, (tr.SCHED_DIRECT, 16), (tr.SCHED_COLUMN_PF1, 8)
RULE = [
    ((512, 512, 512), (TILE, 512)),
    ((512, 512, 300), (TILE, 512)),    # one round of 300 planes
    ((512, 512, 64), (TILE, 512)),
    ((512, 512, 10), (TILE, 512)),
    ((512, 512, 9), DIRECT),           # too thin
    ((500, 512, 100), (TILE, 512)),
    ((256, 512, 200), (TILE, 128)),    # one round of 128 planes, the second chunk of 72: 0.78
    ((512, 384, 512), (TILE, 256)),    # 384 workgroups, 0.75
    ((384, 512, 200), WAVE),           # 384 workgroups of 128 planes, 0.59
    ((2048, 2048, 4), WAVE),
    ((160, 160, 160), DIRECT),
]


@pytest.mark.parametrize("box,schedule", RULE)
def test_schedule_of_a_box(box, schedule):
    tr.tune()
    assert tr.schedule(nh.Layout.build(box, 1)) == schedule


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(512, 512, 10), (512, 512, 9), (390, 512, 70), (48, 40, 36)])
@pytest.mark.parametrize("stage", [1, 2, 3])
def test_bits_of_every_choice(n, stage):
    import torch
    L = nh.Layout.build(n, 1)
    faces = [L.like(f) for f in ("SSurfX", "SSurfY", "SSurfZ")]
    c = nh.axis_coefs(nh.build_stencils(*n, 1.0, 1.0, 1.0))
    g = torch.Generator("cuda").manual_seed(sum(n) + stage)
    rand = lambda: torch.rand(L.npts, generator=g, device="cuda", dtype=torch.float64)
    pn, s, a, acc, k = rand(), rand(), rand(), rand(), rand() + 0.5
    u = [rand() - 0.5 for _ in range(3)]
    gk0 = rand()
    got = []
    for schedule in (0, 1):
        tr.tune(schedule, 0)
        try:
            out, lam, acc2, gk = (torch.zeros_like(pn) for _ in range(4))
            gk.copy_(gk0)
            tr.stage(L, out, pn, None if stage == 1 else s, k, u, c, 1e-6, stage, faces)
            tr.adjoint_stage(L, lam, None if stage == 1 else acc2, gk, a, None if stage == 3 else acc, s, k, u, c, 1e-6,
                             stage, faces)
            torch.cuda.synchronize()
            got.append((out, lam, acc2, gk))
        finally:
            tr.tune()
    for x, y in zip(*got):
        assert torch.equal(x, y)
