"""ParticleToCell of particles in an order of space: each block of the count then has many
records in one brick, which one wave writes in parts of 64 particles.  Parts that end
inside a block, blocks of fewer than 64 particles, parts whose particles all reach one
brick, particles that are skipped or reach no cell in between, and sets crowded past
the line to the sort.  Bar: the oracle's bits."""
import numpy as np
import pytest
import torch

import nebo_hip as nh
from nebo_hip import particles as P
import oracle_lib as orc

pytestmark = pytest.mark.gpu

ORDERS = {"cell": 1, "block": 8, "plane": 64}


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to("cuda:0")


def check(n, coords, size, src):
    L = nh.Layout.build(n, 1)
    cells = nh.Field.from_numpy(L, np.random.default_rng(1).standard_normal(L.npts), where="both")
    geom = (1.0, 0.5, 1.0, 0.5, 1.0, 0.5)
    op = P.ParticleToCell(*geom)
    op.set_coordinate_information(*[dev(c) for c in coords], dev(size))
    op.apply_to_field(dev(src), cells)
    orc.particle_to_cell(cells, src, *coords, size, geom)
    torch.cuda.synchronize()
    assert np.array_equal(cells.gpu.cpu().numpy(), cells.host)


def ordered(n, npart, order, seed, beyond=0.0):
    rng = np.random.default_rng(seed)
    coords = [rng.uniform(-beyond, e + beyond, npart) for e in n]
    key = [np.floor(c / ORDERS[order]).astype(np.int64) for c in coords]
    at = np.lexsort((key[0], key[1], key[2]))
    return [c[at] for c in coords], rng.uniform(0.2, 1.5, npart), rng.standard_normal(npart)


@pytest.mark.parametrize("order", ORDERS)
@pytest.mark.parametrize("n,npart", [((24, 24, 24), 5000), ((64, 64, 64), 20000), ((50, 31, 40), 70001),
                                     ((16, 90, 70), 130000), ((100, 90, 80), 521234)])
def test_ordered_particles(n, npart, order):
    check(n, *ordered(n, npart, order, npart))


def test_ordered_particles_some_of_them_outside():
    check((40, 40, 40), *ordered((40, 40, 40), 90000, "cell", 7, beyond=3.0))


@pytest.mark.parametrize("npart", [33, 63, 64, 65, 127, 129, 500, 1025])
def test_all_particles_in_one_brick(npart):
    rng = np.random.default_rng(npart)
    check((64, 64, 64), [rng.uniform(17.2, 18.8, npart) for _ in range(3)], rng.uniform(0.2, 0.9, npart),
          rng.standard_normal(npart))


@pytest.mark.parametrize("order", ORDERS)
@pytest.mark.parametrize("share,width", [(0.02, 3.0), (0.2, 20.0), (0.5, 4.0)])
def test_ordered_and_crowded(order, share, width):
    n, npart = (64, 64, 64), 60000
    rng = np.random.default_rng(int(100 * share))
    coords = [rng.uniform(0.0, e, npart) for e in n]
    for c in coords:
        c[:int(share * npart)] = 20.0 + rng.uniform(0.0, width, int(share * npart))
    key = [np.floor(c / ORDERS[order]).astype(np.int64) for c in coords]
    at = np.lexsort((key[0], key[1], key[2]))
    check(n, [c[at] for c in coords], rng.uniform(0.2, 1.5, npart), rng.standard_normal(npart))
