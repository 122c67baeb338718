"""Particles whose cell range leaves 32-bit arithmetic: cubes of negative size (empty
ranges in the reference's loops), coordinates far past the window, and values that
overflow, among ordinary particles.  Bar: the oracle's bits."""
import numpy as np
import pytest
import torch

import nebo_hip as nh
from nebo_hip import particles as P
import oracle_lib as orc

pytestmark = pytest.mark.gpu

GEOM = (1.0, 0.5, 1.0, 0.5, 1.0, 0.5)
# (coordinate on every axis, size): the low face lies |size| / 2 above a particle of
# negative size, so its first cell is far past its last
ODD = [(5.0, -1.0), (5.0, -3.0e8), (5.0, -4.0e9), (5.0, -1.0e10), (5.0, -7.0e15), (-2.0, -6.0e9),
       (1.0e10, 0.5), (1.0e15, 1.0), (3.0, 1.0e10), (4.5e9, 9.0e9 - 4.0), (3.0e9, -3.0e9)]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to("cuda:0")


@pytest.mark.parametrize("axes", [(0,), (0, 1), (0, 1, 2)])
def test_ranges_past_32_bits(axes):
    n = tuple(13 if a in axes else 1 for a in range(3))
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(len(axes))
    m = 300
    size = rng.uniform(0.2, 1.5, m)
    coords = [rng.uniform(0.0, 13.0, m) if a in axes else None for a in range(3)]
    for i, (x, s) in enumerate(ODD):
        at = 7 + 25 * i
        size[at] = s
        for a in axes:
            coords[a][at] = x
    geom = tuple(v for a in range(3) for v in (GEOM[2 * a:2 * a + 2] if a in axes else (-1.0, 0.0)))
    src = rng.standard_normal(m)
    cells = nh.Field.from_numpy(L, rng.standard_normal(L.npts), where="both")
    on_gpu = [None if c is None else dev(c) for c in coords]
    c2p, p2c = P.CellToParticle(*geom), P.ParticleToCell(*geom)
    for op in (c2p, p2c):
        op.set_coordinate_information(*on_gpu, dev(size))
    out = c2p.apply_to_field(cells, torch.full((m,), 9.0, dtype=torch.float64, device="cuda:0"))
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        want = orc.cell_to_particle(cells, *coords, size, geom, m)
    assert np.array_equal(out.cpu().numpy(), want, equal_nan=True)
    p2c.apply_to_field(dev(src), cells)
    orc.particle_to_cell(cells, src, *coords, size, geom)
    torch.cuda.synchronize()
    assert np.array_equal(cells.gpu.cpu().numpy(), cells.host, equal_nan=True)


@pytest.mark.parametrize("mask", range(8))
def test_every_set_of_resolved_axes(mask):
    """Axes the particles do not resolve, on a window of several cells along them."""
    n = (9, 8, 7)
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(40 + mask)
    m = 2000
    size = rng.uniform(0.2, 4.0, m)
    coords = [rng.uniform(-1.0, n[a] + 1.0, m) if mask >> a & 1 else None for a in range(3)]
    cells = nh.Field.from_numpy(L, rng.standard_normal(L.npts), where="both")
    op = P.CellToParticle(*GEOM)
    op.set_coordinate_information(*[None if c is None else dev(c) for c in coords], dev(size))
    skipped = torch.zeros(1, dtype=torch.int32, device="cuda:0")
    out = op.apply_to_field(cells, torch.full((m,), 9.0, dtype=torch.float64, device="cuda:0"), skipped=skipped)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), orc.cell_to_particle(cells, *coords, size, GEOM, m))
    # skipped: a cell or more below the window (face -1.0) on some axis
    low = [(c - size * 0.5 + 1.0) / 1.0 for c in coords if c is not None]
    assert skipped.item() == (int(np.any([t <= -1.0 for t in low], axis=0).sum()) if low else 0)
