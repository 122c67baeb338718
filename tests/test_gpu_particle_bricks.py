"""ParticleToCell by bricks where it can go wrong: windows that end inside a brick,
one to three resolved axes, particles larger than a brick, bricks whose records fill
several rounds, and sets too crowded for the path (sorted instead).  Bar: the
oracle's bits."""
import numpy as np
import pytest
import torch

import nebo_hip as nh
from nebo_hip import particles as P
import oracle_lib as orc

pytestmark = pytest.mark.gpu


def dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to("cuda:0")


def scatter(L, src, coords, size, geom):
    cells = nh.Field.from_numpy(L, np.random.default_rng(1).standard_normal(L.npts), where="both")
    skipped = torch.zeros(1, dtype=torch.int32, device="cuda:0")
    op = P.ParticleToCell(*geom)
    op.set_coordinate_information(*[dev(c) for c in coords], dev(size))
    op.apply_to_field(dev(src), cells, skipped=skipped)
    orc.particle_to_cell(cells, src, *coords, size, geom)
    torch.cuda.synchronize()
    assert np.array_equal(cells.gpu.cpu().numpy(), cells.host)
    return skipped.item()


def cloud(rng, n, box, size_lo, size_hi, beyond=0.0):
    size = rng.uniform(size_lo, size_hi, n)
    coords = [None if b is None else rng.uniform(b[0] - beyond, b[1] + beyond, n) for b in box]
    return rng.standard_normal(n), coords, size


@pytest.mark.parametrize("n", [(8, 8, 8), (9, 7, 5), (17, 33, 3), (40, 1, 1), (1, 65, 18), (70, 50, 31)])
@pytest.mark.parametrize("npart", [3, 5000])
def test_windows_that_end_inside_a_brick(n, npart):
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(npart + n[0])
    box = [(0.0, float(e)) if e > 1 else None for e in n]
    geom = tuple(v for e in n for v in ((1.0, 0.5) if e > 1 else (-1.0, 0.0)))
    below = scatter(L, *cloud(rng, npart, box, 0.1, 1.6, beyond=3.0), geom)
    assert below > 0 or npart == 3


# Blocks of counting particles (one per 1024, up to 512, or more where the bricks are
# few), whose counts are summed in 64 parts: one row per part, a last part that is
# full, cut, and empty, and parts longer than one batch of loads.
@pytest.mark.parametrize("npart", [64 * 1024, 65 * 1024, 126 * 1024, 127 * 1024 - 5, 128 * 1024, 443 * 1024 - 7,
                                   511 * 1024 + 1, 600 * 1024, 760 * 1024, 1500 * 1024])
def test_counts_of_every_number_of_blocks(npart):
    n = (50, 70, 36)
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(npart)
    scatter(L, *cloud(rng, npart, [(0.0, float(e)) for e in n], 0.2, 1.2, beyond=0.5), (1.0, 0.5, 1.0, 0.5, 1.0, 0.5))


@pytest.mark.parametrize("edge", [0.0, 1.0, 6.5, 30.0])
def test_particles_of_every_size(edge):
    """Cubes of no volume (0/0 in the reference too), of whole cells, wider than a
    brick and wider than the window."""
    L = nh.Layout.build((21, 19, 23), 2)
    rng = np.random.default_rng(int(edge * 2))
    src, coords, _ = cloud(rng, 400, [(0.0, 21.0), (0.0, 19.0), (0.0, 23.0)], 1.0, 1.0)
    if edge == 1.0:
        coords = [np.floor(c) + 0.5 for c in coords]
    size = np.full(400, edge)
    cells = nh.Field.from_numpy(L, np.zeros(L.npts), where="both")
    geom = (1.0, 0.5, 1.0, 0.5, 1.0, 0.5)
    op = P.ParticleToCell(*geom)
    op.set_coordinate_information(*[dev(c) for c in coords], dev(size))
    op.apply_to_field(dev(src), cells)
    orc.particle_to_cell(cells, src, *coords, size, geom)
    torch.cuda.synchronize()
    assert np.array_equal(cells.gpu.cpu().numpy(), cells.host, equal_nan=True)


@pytest.mark.parametrize("npart", [31, 32, 33, 12000, 140000])
def test_one_crowded_brick(npart):
    """All particles in two cells per axis of a wide window: 32 records of one block in
    one brick, and 131072 records in one brick, are the path's limits."""
    L = nh.Layout.build((64, 64, 64), 1)
    rng = np.random.default_rng(npart)
    src, coords, size = cloud(rng, npart, [(8.9, 9.1), (9.0, 9.9), (17.6, 18.4)], 0.2, 0.9)
    scatter(L, src, coords, size, (1.0, 0.5, 1.0, 0.5, 1.0, 0.5))


def test_dense_and_empty_bricks_together():
    L = nh.Layout.build((50, 60, 40), 1)
    rng = np.random.default_rng(77)
    a = cloud(rng, 30000, [(0.0, 12.0), (30.0, 41.0), (0.0, 9.0)], 0.2, 1.5)
    b = cloud(rng, 500, [(0.0, 50.0), (0.0, 60.0), (0.0, 40.0)], 0.2, 5.0)
    mix = rng.permutation(30500)
    scatter(L, np.concatenate([a[0], b[0]])[mix], [np.concatenate([x, y])[mix] for x, y in zip(a[1], b[1])],
            np.concatenate([a[2], b[2]])[mix], (1.0, 0.5, 1.0, 0.5, 1.0, 0.5))


@pytest.mark.parametrize("axes", [(0,), (1, 2), (0, 1, 2)])
@pytest.mark.parametrize("edge,spacing", [((0.2, 1.5), (1.0, 1.0, 1.0)), ((1.0, 1.0), (1.0, 1.0, 1.0)),
                                          ((2.5, 4.5), (0.3, 0.7, 1.1)), ((0.2, 2.0), (3e-151, 3e-151, 3e-151)),
                                          ((0.2, 2.0), (1e140, 1e140, 1e140)), ((0.0, 0.0), (1.0, 1.0, 1.0))])
def test_gather_of_every_span(axes, edge, spacing):
    """CellToParticle of particles of up to three cells per axis and more, with faces on
    cell faces, and with spacings whose products leave the range of the fast quotient."""
    n = tuple(17 if a in axes else 1 for a in range(3))
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(int(10 * edge[1]) + len(axes))
    m = 3000
    unit = rng.uniform(*edge, m)
    size = unit * min(spacing[a] for a in axes)
    coords = [None] * 3
    for a in axes:
        x = rng.uniform(-2.0, 19.0, m)
        x[::3] = np.floor(x[::3]) + unit[::3] / 2      # the low face on a cell face
        coords[a] = x * spacing[a]
    geom = tuple(v for a in range(3) for v in ((spacing[a], 0.5 * spacing[a]) if a in axes else (-1.0, 0.0)))
    cells = nh.Field.from_numpy(L, rng.standard_normal(L.npts), where="both")
    op = P.CellToParticle(*geom)
    op.set_coordinate_information(*[dev(c) for c in coords], dev(size))
    skipped = torch.zeros(1, dtype=torch.int32, device="cuda:0")
    out = op.apply_to_field(cells, torch.full((m,), 9.0, dtype=torch.float64, device="cuda:0"), skipped=skipped)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        want = orc.cell_to_particle(cells, *coords, size, geom, m)
    assert np.array_equal(out.cpu().numpy(), want, equal_nan=True)
    assert skipped.item() > 0


@pytest.mark.parametrize("n,npart", [((16, 16, 16), 1000), ((24, 24, 24), 5000), ((32, 32, 32), 20000),
                                     ((160, 30, 10), 300), ((60, 50, 40), 20000), ((16, 16, 16), 20000),
                                     ((100, 60, 1), 60000), ((12, 12, 12), 8000)])
def test_brick_sizes_and_the_line_to_the_sort(n, npart):
    """Rows of fewer than 1024 particles, bricks of 64 to 1024 cells, and sets on both
    sides of the line past which they are sorted."""
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(npart + n[0])
    box = [(0.0, float(e)) for e in n]
    scatter(L, *cloud(rng, npart, box, 0.2, 1.5), (1.0, 0.5, 1.0, 0.5, 1.0, 0.5))
