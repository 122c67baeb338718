"""Periodic chains (diffusion and transport steps and their transposes) on boxes at
the edges of their schedules: axes of one, two and three cells, widths around a wave,
each rule of the size choice.  The kernels write the ghost images of their output
themselves, so whole blocks are compared.  Bar: the oracle's bits."""
import numpy as np
import pytest
import torch

import nebo_hip as nh
from nebo_hip import adjoint as adj
from nebo_hip import transport as tr
import oracle_lib as orc

pytestmark = pytest.mark.gpu

# direct (4 x 2 planes; 16 planes), 2 rows x 4 planes, 2 rows x 8 planes, and (transpose)
# more waves than 28 per CU
BOXES = [(1, 1, 1), (1, 5, 2), (2, 1, 3), (3, 2, 1), (2, 2, 2), (63, 3, 5), (64, 2, 17), (65, 7, 4), (64, 64, 64),
         (129, 10, 33), (100, 90, 33), (66, 130, 67)]


def layout(n):
    """One ghost layer on every axis, those of one cell included (Layout.build gives
    such axes none)."""
    e = tuple(v + 2 for v in n)
    one, none = (1, 1, 1), (0, 0, 0)
    return nh.Layout(glob=e, offset=none, extent=e, ghost_minus=one, ghost_plus=one, valid_minus=one, valid_plus=one,
                     has_bc=none, bc_extra=none)


def block(n, rng, lo=-1.0, hi=1.0):
    return np.pad(rng.uniform(lo, hi, n[::-1]), 1, mode="wrap").reshape(-1)


def dev(a):
    return torch.from_numpy(a).cuda()


def same(t, want):
    torch.cuda.synchronize()
    return np.array_equal(t.cpu().numpy(), want)


@pytest.mark.parametrize("n", BOXES)
def test_diffusion_step_and_transpose(n):
    L, rng = layout(n), np.random.default_rng(sum(n))
    c = nh.axis_coefs(nh.build_stencils(7, 11, 13, 1.0, 1.0, 1.0))
    phi, lam, k = block(n, rng), block(n, rng), block(n, rng, 0.5, 2.0)
    zero, g0 = np.zeros(L.npts), rng.standard_normal(L.npts)
    want, wl, wg = nh.Field(L, host=zero.copy()), nh.Field(L, host=zero.copy()), g0.copy()
    orc.diffusion_step(want, nh.Field(L, host=phi), nh.Field(L, host=k), c, 1e-4)
    orc.diffusion_adjoint_step(wl, wg, nh.Field(L, host=lam), nh.Field(L, host=phi), nh.Field(L, host=k), c, 1e-4)
    out, lo, gk = dev(zero), dev(zero), dev(g0)
    adj.diffusion_step(L, out, dev(phi), dev(k), c, 1e-4)
    adj.diffusion_adjoint_step(L, lo, gk, dev(lam), dev(phi), dev(k), c, 1e-4)
    assert same(out, want.host)
    assert same(lo, wl.host) and same(gk, wg)


@pytest.mark.parametrize("n", BOXES)
def test_transport_stage_and_transpose(n):
    L, rng = layout(n), np.random.default_rng(sum(n) + 1)
    c = nh.axis_coefs(nh.build_stencils(7, 11, 13, 1.0, 1.0, 1.0))
    pn, s, a, acc = (block(n, rng) for _ in range(4))
    k, u = block(n, rng, 0.5e-3, 2e-3), [block(n, rng) for _ in range(3)]
    inner = np.zeros(L.glob[::-1], dtype=bool)
    inner[1:-1, 1:-1, 1:-1] = True
    inner, faces = inner.reshape(-1), [L] * 3
    hu = [nh.Field(L, host=x) for x in u]
    gu, gpn, gs, ga, gacc, gk_ = [dev(x) for x in u], dev(pn), dev(s), dev(a), dev(acc), dev(k)
    for stage in (1, 2, 3):
        want = nh.Field(L, host=np.zeros(L.npts))
        orc.transport_stage(want, nh.Field(L, host=pn), nh.Field(L, host=s if stage != 1 else pn),
                            nh.Field(L, host=k), hu, c, 1e-3, stage)
        out = torch.zeros_like(gpn)
        tr.stage(L, out, gpn, gs if stage != 1 else None, gk_, gu, c, 1e-3, stage, face_layouts=faces)
        assert same(out, want.host), stage
        wo, wacc, wg = nh.Field(L, host=np.zeros(L.npts)), np.zeros(L.npts), np.full(L.npts, 0.5)
        orc.transport_adjoint_stage(wo, wacc if stage != 1 else None, wg, nh.Field(L, host=a),
                                    acc if stage != 3 else None, nh.Field(L, host=s), nh.Field(L, host=k), hu, c,
                                    1e-3, stage)
        o, ao, g = torch.zeros_like(gpn), torch.zeros_like(gpn), dev(np.full(L.npts, 0.5))
        tr.adjoint_stage(L, o, ao if stage != 1 else None, g, ga, gacc if stage != 3 else None, gs, gk_, gu, c, 1e-3,
                         stage, face_layouts=faces)
        assert same(o, wo.host) and same(g, wg), stage
        assert stage == 1 or same(ao[dev(inner)], wacc[inner]), stage


@pytest.mark.parametrize("ghost", [((1, 1, 1), (1, 1, 1)), ((2, 0, 1), (0, 3, 2)), ((3, 3, 3), (3, 3, 3))])
@pytest.mark.parametrize("n", [(3, 4, 5), (70, 3, 6)])
def test_ghost_fill_of_uneven_layers(n, ghost):
    L = nh.Layout.build(n, ghost)
    f = nh.Field.from_numpy(L, np.random.default_rng(1).standard_normal(L.npts))
    nh.fill_ghosts_periodic(f)
    orc.fill_periodic(f)
    assert same(f.gpu, f.host)


@pytest.mark.parametrize("n", [(112, 150, 130), (256, 128, 100)])
def test_diffusion_step_of_8_and_16_planes(n):
    """Boxes on which the size rule gives 16 planes and the step takes 8, and 16."""
    L, rng = layout(n), np.random.default_rng(sum(n))
    c = nh.axis_coefs(nh.build_stencils(7, 11, 13, 1.0, 1.0, 1.0))
    phi, k, zero = block(n, rng), block(n, rng, 0.5, 2.0), np.zeros(L.npts)
    want, out = nh.Field(L, host=zero.copy()), dev(zero)
    orc.diffusion_step(want, nh.Field(L, host=phi), nh.Field(L, host=k), c, 1e-4)
    adj.diffusion_step(L, out, dev(phi), dev(k), c, 1e-4)
    assert nh.stencil_select_tile(0, n) == (64, 2, 16, 3)
    assert same(out, want.host)
