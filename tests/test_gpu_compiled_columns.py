"""Column kernels of the run-time compiler whose reads on one x side lie on
several rows or planes: each value from the adjacent lane is formed once and
kept while a cell of the lane still reads it.  Against the oracle, bit for bit.
"""
import numpy as np
import pytest

import nebo_hip as nh
import oracle_lib as orc
from test_gpu_parity import both, fetch, gpu_empty_like

pytestmark = pytest.mark.gpu

COEF = [0.37, -1.21, 0.83, 2.09, -0.55, 1.31, 0.19, -0.71, 0.97]


def _trees(L, phi, k, n):
    filt = nh.build_stencils(*n, 1.0, 1.0, 1.0)[("Filter", "SVol", "SVol")]
    square = nh.Stencil([(x, y, 0) for y in (-1, 0, 1) for x in (-1, 0, 1)], COEF)
    upright = nh.Stencil([(x, 0, z) for z in (-1, 0, 1) for x in (-1, 0, 1)], COEF)
    right_rows = nh.Stencil([(0, 0, 0), (1, 0, 0), (1, 1, 0)], COEF[:3])
    left_planes = nh.Stencil([(0, 0, 0), (-1, 0, 0), (-1, 0, 1)], COEF[:3])
    slanted = nh.Stencil([(-1, 0, -1), (-1, 1, 0), (0, 0, 0), (1, 0, 1), (1, -1, 0)], COEF[:5])
    return {"filter": filt(phi), "square": square(phi), "upright": upright(phi), "right_rows": right_rows(phi),
            "left_planes": left_planes(phi), "slanted": slanted(phi),
            "two_fields": filt(phi) * k + square(k) * phi, "two_sided": right_rows(k) * left_planes(phi) - slanted(k)}


@pytest.mark.parametrize("column", [(1, 0, 0), (1, 1, 3), (1, 2, 64), (2, 3, 5)],
                         ids=["default", "w1-z3", "w2-z64", "one-column-w3-z5"])
@pytest.mark.parametrize("n", [(100, 37, 21), (131, 9, 10), (64, 5, 2)])
def test_shared_neighbours_match_oracle(column, n):
    L = nh.Layout.build(n, 2)
    rng = np.random.default_rng(29)
    phi, k = both(L, rng.standard_normal(L.npts)), both(L, rng.uniform(0.5, 2.0, L.npts))
    try:
        nh.fused_jit_column(*column)
        for name, t in _trees(L, phi, k, n).items():
            for use_ghost in (True, False):
                print(f"{n} column {column} {name} use_ghost={use_ghost}", flush=True)
                out = gpu_empty_like(L, 7.0)
                ref = nh.Field.from_numpy(L, np.full(L.npts, 7.0), where="cpu")
                nh.assign(out, t, use_ghost=use_ghost, generic=True)
                orc.assign(ref, t, use_ghost=use_ghost)
                assert np.array_equal(fetch(out), ref.host), (column, name, use_ghost)
    finally:
        nh.fused_jit_column()


def _few_reads(L, phi, k):
    """Three fields at 2 reads each."""
    g = both(L, np.random.default_rng(31).standard_normal(L.npts))
    lo = nh.Stencil([(0, 0, -1), (0, 0, 0)], COEF[:2])
    side = nh.Stencil([(-1, 0, 0), (0, 0, 0)], COEF[1:3])
    return lo(phi) * side(k) + lo(g)


# Boxes of every planes-per-block choice, of one and two columns per lane, and on both
# sides of the line where trees of few reads leave the schedule.
@pytest.mark.parametrize("n,few_flat", [((40, 36, 30), True), ((100, 90, 20), True), ((180, 50, 70), True),
                                        ((130, 129, 131), False), ((300, 200, 33), False)])
def test_default_schedule_matches_oracle(n, few_flat):
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(37)
    phi, k = both(L, rng.standard_normal(L.npts)), both(L, rng.uniform(0.5, 2.0, L.npts))
    trees = {x: t for x, t in _trees(L, phi, k, n).items() if x in ("filter", "two_fields", "two_sided")}
    for name, t in {**trees, "few_reads": _few_reads(L, phi, k)}.items():
        print(f"{n} {name}", flush=True)
        out = gpu_empty_like(L, 7.0)
        ref = nh.Field.from_numpy(L, np.full(L.npts, 7.0), where="cpu")
        nh.assign(out, t, use_ghost=False, generic=True)
        assert ("column schedule" in nh.last_backend()) == (name != "few_reads" or not few_flat), nh.last_backend()
        orc.assign(ref, t, use_ghost=False)
        assert np.array_equal(fetch(out), ref.host), (name, nh.last_backend())


# Boxes of 1, 2 and 4 cells per thread, with planes below and past one block and z
# extents that cut the last cells.
@pytest.mark.parametrize("n,masked_cells", [((5, 3, 2), 1), ((33, 31, 30), 1), ((129, 90, 50), 2),
                                            ((160, 131, 111), 4)])
def test_flattened_shapes_match_oracle(n, masked_cells):
    L = nh.Layout.build(n, 1)
    rng = np.random.default_rng(41)
    phi, k = both(L, rng.standard_normal(L.npts)), both(L, rng.uniform(0.5, 2.0, L.npts))
    m = nh.Mask(L, [(x, y, n[2] - 1) for x in range(n[0]) for y in range(0, n[1], 2)]).add_consumer(0)
    for name, t in {"masked": nh.cond(m, 0.25)(phi), "two": 0.5 * phi + k}.items():
        for use_ghost in (True, False):
            out = gpu_empty_like(L, 7.0)
            ref = nh.Field.from_numpy(L, np.full(L.npts, 7.0), where="cpu")
            nh.assign(out, t, use_ghost=use_ghost, generic=True)
            cells = masked_cells if name == "masked" else min(masked_cells, 2)
            assert f"{cells} z cells per thread (256-thread blocks)" in nh.last_backend(), nh.last_backend()
            orc.assign(ref, t, use_ghost=use_ghost)
            assert np.array_equal(fetch(out), ref.host), (name, use_ghost, nh.last_backend())
