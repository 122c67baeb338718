"""Assignments whose limits leave the field's block (fewer valid ghosts than ghosts) are
refused before anything is launched; those that stay inside are not."""
import numpy as np
import pytest

import nebo_hip as nh


def field(L):
    return nh.Field.from_numpy(L, np.zeros(L.npts), where="cpu")


@pytest.mark.parametrize("minus,plus", [((1, 2, 2), (2, 2, 2)), ((2, 2, 2), (2, 2, 0)), ((2, 0, 2), (2, 1, 2)),
                                        ((0, 0, 0), (0, 0, 0))])
def test_cells_outside_the_block_are_refused(minus, plus):
    L = nh.Layout.build((7, 6, 5), 2)
    out, f = field(L.with_valid(minus, plus)), field(L)
    for rhs in (0.0, nh.E(f) + 1.0):
        with pytest.raises(nh.NeboError, match="outside the field's block"):
            nh.assign_limits(out, rhs, True, where="host")
    # the interior, and what operands with the same valid ghosts give
    inside = nh.assign_limits(out, 0.0, False, where="host")
    assert inside == ((0, 0, 0), tuple(e - a - b for e, a, b in zip(L.extent, minus, plus)))
    assert nh.assign_limits(out, nh.E(field(L.with_valid(minus, plus))) * 2.0, True, where="host") == \
        (tuple(-m for m in minus), tuple(e - m for e, m in zip(L.extent, minus)))


def test_a_window_inside_a_larger_block_is_not_refused():
    W = nh.Layout(glob=(13, 12, 11), offset=(1, 1, 1), extent=(11, 10, 9), ghost_minus=(2,) * 3, ghost_plus=(2,) * 3,
                  valid_minus=(1,) * 3, valid_plus=(1,) * 3, has_bc=(0,) * 3, bc_extra=(0,) * 3)
    assert nh.assign_limits(field(W), 0.0, True, where="host") == ((-2, -2, -2), (11, 10, 9))


@pytest.mark.parametrize("bc", [(False,) * 3, (True,) * 3])
@pytest.mark.parametrize("loc", ["SVol", "SSurfX", "XVol"])
def test_ordinary_fields_are_not_refused(loc, bc):
    for ghost in (0, 1, 3):
        for n in ((7, 6, 5), (7, 1, 5), (1, 1, 4)):
            L = nh.Layout.build(n, ghost, loc, bc)
            lo, hi = nh.assign_limits(field(L), 0.0, True, where="host")
            assert all(h - l == g for l, h, g in zip(lo, hi, L.glob))
