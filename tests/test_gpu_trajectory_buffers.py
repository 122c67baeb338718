"""Trajectories and their reverse sweeps against the same steps and transposes called one
by one: odd and even numbers of steps (lam goes back and forth between two blocks),
segments of one step and more, inputs whose ghost cells hold anything, and a window
inside a larger block.  Bar: the same bits."""
import numpy as np
import pytest
import torch

import nebo_hip as nh
from nebo_hip import adjoint as adj
from nebo_hip import transport as tr

pytestmark = pytest.mark.gpu


def layout(n, around=0):
    e, one, none = tuple(v + 2 for v in n), (1, 1, 1), (0, 0, 0)
    return nh.Layout(glob=tuple(v + around for v in e), offset=(around // 2,) * 3, extent=e, ghost_minus=one,
                     ghost_plus=one, valid_minus=one, valid_plus=one, has_bc=none, bc_extra=none)


def window(L, t):
    g, o, e = L.glob, L.offset, L.extent
    return t.reshape(g[2], g[1], g[0])[o[2]:o[2] + e[2], o[1]:o[1] + e[1], o[0]:o[0] + e[0]]


def wrapped(L, t):
    """t with its ghost cells the images of its interior."""
    t = t.clone()
    w = window(L, t)
    for a in range(3):
        w.select(a, 0).copy_(w.select(a, -2))
        w.select(a, w.shape[a] - 1).copy_(w.select(a, 1))
    return t


def same(L, a, b):
    return torch.equal(window(L, a), window(L, b))


CASES = [((5, 4, 3), 1, 1, 0), ((9, 1, 6), 2, 1, 0), ((70, 9, 6), 3, 3, 0), ((12, 11, 10), 4, 2, 3),
         ((66, 20, 33), 6, 3, 2)]


@pytest.mark.parametrize("n,steps,every,around", CASES)
def test_diffusion(n, steps, every, around):
    L, dt = layout(n, around), 1e-4
    g = torch.Generator("cuda").manual_seed(sum(n) + steps)
    rand = lambda: torch.rand(L.npts, generator=g, device="cuda", dtype=torch.float64)
    c = nh.axis_coefs(nh.build_stencils(7, 11, 13, 1.0, 1.0, 1.0))
    phi0, lamT, k = rand(), rand(), wrapped(L, rand() + 0.5)
    end, ckpt = adj.forward(L, phi0, k, c, dt, steps, every)
    lam0, gk = adj.backward(L, lamT, k, c, dt, steps, every, ckpt)
    states = [wrapped(L, phi0)]
    for _ in range(steps):
        states.append(torch.zeros_like(phi0))
        adj.diffusion_step(L, states[-1], states[-2], k, c, dt)
    lam, want = wrapped(L, lamT), torch.zeros_like(gk)
    for t in reversed(range(steps)):
        nxt = torch.zeros_like(lam)
        adj.diffusion_adjoint_step(L, nxt, want, lam, states[t], k, c, dt)
        lam = nxt
    assert same(L, end, states[-1])
    for q in range(steps // every + 1):
        assert same(L, ckpt[q * L.npts:(q + 1) * L.npts], states[q * every])
    assert same(L, lam0, lam) and same(L, gk, want)


@pytest.mark.parametrize("n,steps,every,around", CASES)
def test_transport(n, steps, every, around):
    L, dt = layout(n, around), 1e-3
    g = torch.Generator("cuda").manual_seed(sum(n) + steps)
    rand = lambda: torch.rand(L.npts, generator=g, device="cuda", dtype=torch.float64)
    c = nh.axis_coefs(nh.build_stencils(7, 11, 13, 1.0, 1.0, 1.0))
    phi0, lamT, k = rand(), rand(), wrapped(L, rand() * 1e-3)
    u, faces = [wrapped(L, rand() - 0.5) for _ in range(3)], [L, L, L]
    end, ckpt = tr.forward(L, phi0, k, u, c, dt, steps, every, face_layouts=faces)
    lam0, gk = tr.backward(L, lamT, k, u, c, dt, steps, every, ckpt, face_layouts=faces)
    states, zero = [wrapped(L, phi0)], torch.zeros_like(phi0)
    kept = []
    for _ in range(steps):
        p, s1, s2, q = states[-1], zero.clone(), zero.clone(), zero.clone()
        tr.stage(L, s1, p, p, k, u, c, dt, 1, face_layouts=faces)
        tr.stage(L, s2, p, s1, k, u, c, dt, 2, face_layouts=faces)
        tr.stage(L, q, p, s2, k, u, c, dt, 3, face_layouts=faces)
        kept.append((p, s1, s2))
        states.append(q)
    lam, want = wrapped(L, lamT), torch.zeros_like(gk)
    for p, s1, s2 in reversed(kept):
        m2, m1, nxt, acc, acc2 = (torch.zeros_like(lam) for _ in range(5))
        tr.adjoint_stage(L, m2, acc, want, lam, None, s2, k, u, c, dt, 3, face_layouts=faces)
        tr.adjoint_stage(L, m1, acc2, want, m2, acc, s1, k, u, c, dt, 2, face_layouts=faces)
        tr.adjoint_stage(L, nxt, None, want, m1, acc2, p, k, u, c, dt, 1, face_layouts=faces)
        lam = nxt
    assert same(L, end, states[-1])
    for q in range(steps // every + 1):
        assert same(L, ckpt[q * L.npts:(q + 1) * L.npts], states[q * every])
    assert same(L, lam0, lam) and same(L, gk, want)
