"""What the generic evaluator launches for an assignment, as a GPU of 256 compute units
has it: the address audit of test_fused_addresses on the schedules chosen by the box
(2 and 4 planes per block, fewer rows per lane, one column per lane for trees that could
have two), and the trees and boxes that leave the column schedule."""
import ctypes as C
import tempfile

import numpy as np
import pytest

import nebo_hip as nh
from nebo_hip import _abi
import test_fused_addresses as fa

pytestmark = fa.pytestmark


def assign_launch(lhs, rhs, use_ghost=False):
    """(source, argument bytes, grid, block), and whether it is the column schedule."""
    s = nh.serialize(nh.E(rhs), "host")
    d = lhs.desc("host")
    need, grid, block, column = (C.c_int32() for _ in range(4))
    args = C.create_string_buffer(1280)
    tail = (args, 1280, C.byref(grid), C.byref(block), C.byref(column))
    _abi.call("nebo_fused_assign_launch", C.byref(d), s.ref, int(use_ghost), None, 0, C.byref(need), *tail)
    buf = C.create_string_buffer(need.value)
    _abi.call("nebo_fused_assign_launch", C.byref(d), s.ref, int(use_ghost), buf, need.value, C.byref(need), *tail)
    return (buf.value.decode(), args.raw, grid.value, block.value), column.value


def trees(n, L):
    rng = np.random.default_rng(sum(n))
    f, g, h = (fa.host_field(L, c, rng) for c in "fgh")
    db = nh.build_stencils(*n, 1.0, 1.0, 1.0)
    ops = nh.basic_op_types(db)
    divk = sum((ops[f"Div{a}"](ops[f"InterpC2F{a}"](g) * ops[f"Grad{a}"](f)) for a in "YZ"),
               ops["DivX"](ops["InterpC2FX"](g) * ops["GradX"](f)))
    return (f, g, h), {"filter": db[("Filter", "SVol", "SVol")](f), "divk": divk,
                       "few": f + ops["DivX"](ops["GradX"](g) * ops["InterpC2FX"](h)) + ops["DivY"](ops["GradY"](h)),
                       "point": 2.0 * f + g}


# box, tree, blocks, threads: from the rows and planes named
LAUNCHES = [
    ((40, 36, 30), "filter", 36 * 15, 64),              # 1 row per lane, 2 planes
    ((64, 64, 64), "filter", 32 * 32, 64),              # 2 rows, 2 planes
    ((100, 90, 40), "filter", 2 * 23 * 20, 64),         # 4 rows, 2 planes
    ((70, 30, 20), "divk", None, None),                 # two columns per lane, one, and two
    ((190, 100, 50), "divk", None, None),
    ((128, 64, 64), "divk", None, None),
]


def test_chosen_column_kernels_stay_in_bounds():
    jobs, pairs = [], set()
    for n, name, blocks, threads in LAUNCHES:
        for use_ghost in (False, True):
            L = nh.Layout.build(n, 1)
            fields, t = trees(n, L)
            out = nh.Field.empty(L, "cpu", name="out")
            launch, column = assign_launch(out, t[name], use_ghost)
            assert column == 1, (n, name)
            if blocks and not use_ghost:
                assert launch[2:] == (blocks, threads), (n, name, launch[2:])
            if name == "divk":
                pairs.add("ld2_(rs_" in launch[0])
            lim = nh.assign_limits(out, t[name], use_ghost, where="host")
            jobs.append((list(fields) + [out], out, launch, lim, (n, name, use_ghost)))
    assert pairs == {False, True}   # one column per lane, and two
    with tempfile.TemporaryDirectory() as tmp:
        for so, (fields, out, launch, lim, case) in zip(fa.build([j[2][0] for j in jobs], tmp), jobs):
            try:
                fa.audit(so, fields, out, launch, lim)
            except AssertionError as e:
                raise AssertionError(f"{case}: {e}") from None


@pytest.mark.parametrize("n,name,threads", [((40, 36, 30), "few", 256), ((70, 30, 20), "few", 256),
                                            ((40, 36, 30), "point", 256)])
def test_few_reads_and_pointwise_trees_run_flattened(n, name, threads):
    L = nh.Layout.build(n, 1)
    _, t = trees(n, L)
    launch, column = assign_launch(nh.Field.empty(L, "cpu"), t[name])
    assert column == 0 and launch[3] == threads
    assert f"__launch_bounds__({threads})" in launch[0]


def test_the_callers_shape_is_reported():
    L = nh.Layout.build((40, 36, 30), 1)
    _, t = trees((40, 36, 30), L)
    out = nh.Field.empty(L, "cpu")
    try:
        nh.fused_jit_tune(block_threads=128, max_cells=2)
        launch, column = assign_launch(out, t["point"])
        assert (column, launch[3]) == (0, 128)
        nh.fused_jit_column(True, 2, 16)
        launch, column = assign_launch(out, t["filter"])
        assert (column, launch[3]) == (1, 128)
    finally:
        nh.fused_jit_tune()
        nh.fused_jit_column()
