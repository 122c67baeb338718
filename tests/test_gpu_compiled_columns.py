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
