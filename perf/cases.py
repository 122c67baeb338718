"""The work that programs have this engine do, as cases that can be timed.

A case is a plain dict; ``prepare`` makes what a program holds before the call
(fields, operators, descriptors serialised once), ``run`` makes one pass through
the public entry points, ``exact`` computes the same with torch in 64 bits and
``work`` counts what a pass cannot do without.  Boxes are (nx, ny, nz) interior
cells with one ghost layer; everything is fp64, the engine's only type.
"""
import ctypes as C
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "spatialops-threadfix_amd", "python"))
import nebo_hip as nh  # noqa: E402
from nebo_hip import _abi, adjoint, particles, transport  # noqa: E402
from nebo_hip import workloads as W  # noqa: E402
from nebo_hip.batch import Batch  # noqa: E402

DEV = "cuda:0"
F64 = torch.float64


def listed():
    return [
        # The smallest call: a box of one patch, one fused assignment in a host
        # loop over patches; launch and host cost count.
        {"name": "divkgrad_48x40x36", "kind": "divkgrad", "nx": 48, "ny": 40, "nz": 36},
        # One time step of the heat equation example on a 64^3 mesh: Laplacian +
        # Euler, ghost reset through a mask, max and sum for the step's log.
        {"name": "heat_step_64", "kind": "heat", "n": 64},
        # The benchmark expression on the benchmark mesh.
        {"name": "divkgrad_256", "kind": "divkgrad", "nx": 256, "ny": 256, "nz": 256},
        # The same expression on a mesh whose sides suit no tile.
        {"name": "divkgrad_300x210x170", "kind": "divkgrad", "nx": 300, "ny": 210, "nz": 170},
        # A user's own expression, compiled at run time: upwind convection and
        # diffusion of one Euler step, six fields read.
        {"name": "expr_upwind_180x150x130", "kind": "expr", "tree": "upwind", "nx": 180, "ny": 150, "nz": 130},
        # Monitoring: the largest value, the interior norm and a weighted sum.
        {"name": "reduce_200x190x210", "kind": "reduce", "nx": 200, "ny": 190, "nz": 210},
        # Many uneven patches of one process, one launch for all of them.
        {"name": "batch_512", "kind": "batch", "patches": 512, "lo": 16, "hi": 64, "shapes": 5},
        # Gradients through a diffusion trajectory: forward with checkpoints, backward.
        {"name": "diffusion_grad_128", "kind": "diffusion_grad", "nx": 128, "ny": 128, "nz": 128, "steps": 20,
         "every": 5},
        # The largest: one SSP-RK3 step of scalar transport, stage by stage.
        {"name": "transport_step_512", "kind": "transport_step", "nx": 512, "ny": 512, "nz": 512},
        # Gradients through a short transport trajectory on a ragged mesh.
        {"name": "transport_grad_112x96x80", "kind": "transport_grad", "nx": 112, "ny": 96, "nz": 80, "steps": 4,
         "every": 2},
        # Source terms of a particle phase: extensive particle values onto the cells.
        {"name": "particle_to_cell_2m", "kind": "p2c", "nx": 112, "ny": 96, "nz": 104, "particles": 2000000},
        # The gas phase seen by the particles: cell values averaged over each particle.
        {"name": "cell_to_particle_4m", "kind": "c2p", "nx": 128, "ny": 128, "nz": 128, "particles": 4000000},
    ]


KINDS = ("divkgrad", "divkgrad", "heat", "expr", "reduce", "batch", "diffusion_grad", "transport_step",
         "transport_grad", "p2c", "c2p")


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(lo, hi, cells):
        while True:
            b = {"nx": size(lo, hi), "ny": size(lo, hi), "nz": size(lo, hi)}
            if b["nx"] * b["ny"] * b["nz"] <= cells:
                return b

    kind = rng.choice(KINDS)
    if kind == "divkgrad":
        return {"kind": kind, **box(16, 400, 2 ** 24)}
    if kind == "heat":
        return {"kind": kind, "n": size(16, 128)}
    if kind == "expr":
        return {"kind": kind, "tree": rng.choice(("upwind", "reaction", "filter")), **box(24, 300, 2 ** 23)}
    if kind == "reduce":
        return {"kind": kind, **box(16, 300, 2 ** 24)}
    if kind == "batch":
        return {"kind": kind, "patches": size(32, 512), "lo": 16, "hi": rng.randint(24, 64),
                "shapes": rng.randint(1, 10 ** 6)}
    if kind in ("diffusion_grad", "transport_grad"):
        every = rng.randint(1, 5)
        return {"kind": kind, **box(16, 200, 2 ** 21), "steps": every * rng.randint(1, 3), "every": every}
    if kind == "transport_step":
        return {"kind": kind, **box(24, 512, 2 ** 27)}
    return {"kind": kind, **box(16, 160, 2 ** 21), "particles": size(20000, 4000000)}


# ---- inputs ---------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _n(case):
    return (case["nx"], case["ny"], case["nz"])


def _rand(gen, shape, lo, hi):
    return lo + (hi - lo) * torch.rand(shape, generator=gen, device=DEV, dtype=F64)


def _wrap(a):
    """The block of interior a (z, y, x) with one periodic ghost layer."""
    b = torch.empty([s + 2 for s in a.shape], device=DEV, dtype=F64)
    b[1:-1, 1:-1, 1:-1] = a
    b[0], b[-1] = b[-2], b[1]
    b[:, 0], b[:, -1] = b[:, -2], b[:, 1]
    b[:, :, 0], b[:, :, -1] = b[:, :, -2], b[:, :, 1]
    return b


def _waves(n, seed, modes=6):
    """A smooth periodic field: a sum of Fourier modes with wave numbers 1 to 6."""
    rng = random.Random(seed)
    x, y, z = (2 * math.pi * (torch.arange(m, device=DEV, dtype=F64) + 0.5) / m for m in n)
    out = torch.zeros((n[2], n[1], n[0]), device=DEV, dtype=F64)
    for _ in range(modes):
        kx, ky, kz = (rng.randint(1, 6) for _ in range(3))
        a, t = rng.gauss(0.0, 1.0), rng.uniform(0.0, 2 * math.pi)
        out += a * torch.sin((kz * z + t)[:, None, None] + (ky * y)[None, :, None] + (kx * x)[None, None, :])
    return out


def _faces(n, seed):
    """A discretely divergence-free face velocity of both signs, |u| up to 1: each
    component varies along the other two axes only."""
    rng = random.Random(seed)
    x, y, z = (2 * math.pi * (torch.arange(m, device=DEV, dtype=F64) + 0.5) / m for m in n)
    p = [rng.uniform(0.0, 2 * math.pi) for _ in range(6)]
    shape = (n[2], n[1], n[0])
    ux = (torch.sin(z + p[0])[:, None, None] * torch.cos(2 * y + p[1])[None, :, None]).expand(shape)
    uy = (torch.sin(2 * z + p[2])[:, None, None] * torch.cos(x + p[3])[None, None, :]).expand(shape)
    uz = (torch.sin(2 * y + p[4])[None, :, None] * torch.cos(x + p[5])[None, None, :]).expand(shape)
    return [ux, uy, uz]


def _coef(n, seed, scale=1.0):
    return _rand(_gen(seed), (n[2], n[1], n[0]), 0.5 * scale, 2.0 * scale)


def _field(layout, block):
    return nh.Field(layout, gpu=block.reshape(-1))


def _heat_start(n, seed):
    """The heat example's start, its centre and width from the seed; zero ghosts."""
    rng = random.Random(seed)
    x = (torch.arange(n, device=DEV, dtype=F64) + 0.5) / n
    c, s = [rng.uniform(0.4, 0.6) for _ in range(3)], rng.uniform(0.08, 0.12)
    g = [torch.exp(-((x - m) ** 2) / (2 * s * s)) for m in c]
    a = g[2][:, None, None] * g[1][None, :, None] * g[0][None, None, :]
    a = a + 1e-3 * _rand(_gen(seed), a.shape, -1.0, 1.0)
    return torch.nn.functional.pad(a, (1, 1, 1, 1, 1, 1))


def _dims(case):
    rng = random.Random(case["shapes"])
    return [tuple(rng.randint(case["lo"], case["hi"]) for _ in range(3)) for _ in range(case["patches"])]


def _starts(dims):
    """Places of the patches' blocks in one tensor, each on a 256-byte boundary."""
    at, out = 0, []
    for d in dims:
        out.append(at)
        at += -(-(d[0] + 2) * (d[1] + 2) * (d[2] + 2) // 32) * 32
    return out, at


def _particles(case, seed):
    """Positions spread over the box, cube edges of 0.2 to 1.5 cells, unit spacing."""
    g, m = _gen(seed), case["particles"]
    size = _rand(g, m, 0.2, 1.5)
    pos = [size / 2 + (n - size) * torch.rand(m, generator=g, device=DEV, dtype=F64) for n in _n(case)]
    return pos, size, torch.randn(m, generator=g, device=DEV, dtype=F64)


def _diffusion_dt(n):
    return 0.1 / max(n) ** 2 / 2.0


def _transport_dt(n):
    return 0.1 / max(n)


# ---- prepare and run --------------------------------------------------------


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _assign_state(lhs, tree):
    """lhs <<= tree with its descriptors serialised once, as a time loop keeps them."""
    s, d = nh.serialize(nh.E(tree)), lhs.desc("gpu")
    return {"lhs": lhs, "args": (C.byref(d), s.ref), "keep": (s, d, tree)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "heat":
        h = W.HeatStepper(case["n"], slots=1)
        h.fields[0].gpu.copy_(_heat_start(case["n"], seed).reshape(-1))
        return {"run": _run_heat, "stepper": h}
    if kind == "batch":
        dims = _dims(case)
        at, total = _starts(dims)
        a = _rand(_gen(seed), total, -1.0, 1.0)
        b = torch.zeros_like(a)

        def cut(t):
            return [t[o:o + (d[0] + 2) * (d[1] + 2) * (d[2] + 2)] for o, d in zip(at, dims)]

        patches = Batch(cut(a), cut(b), dims, nh.axis_coefs(nh.build_stencils(1, 1, 1, 1.0, 1.0, 1.0)), 0.1)
        patches.autotune()
        b.zero_()
        a.copy_(_rand(_gen(seed), total, -1.0, 1.0))
        return {"run": _run_batch, "batch": patches, "out": b, "keep": a}
    n = _n(case)
    layout = nh.Layout.build(n, 1)
    if kind in ("p2c", "c2p"):
        pos, size, vals = _particles(case, seed)
        geom = (1.0, 0.5, 1.0, 0.5, 1.0, 0.5)
        op = (particles.ParticleToCell if kind == "p2c" else particles.CellToParticle)(*geom)
        op.set_coordinate_information(*pos, size)
        if kind == "p2c":
            return {"run": _run_p2c, "op": op, "src": vals, "dest": _field(layout, torch.zeros(layout.npts, device=DEV, dtype=F64))}
        return {"run": _run_c2p, "op": op, "src": _field(layout, _wrap(_waves(n, seed))), "dest": torch.zeros_like(vals)}
    db = nh.build_stencils(*n, 1.0, 1.0, 1.0)
    ops, coefs = nh.basic_op_types(db), nh.axis_coefs(db)
    phi, k = _wrap(_waves(n, seed)), _wrap(_coef(n, seed))
    if kind in ("divkgrad", "expr", "reduce"):
        fphi, fk = _field(layout, phi), _field(layout, k)
        out = _field(layout, torch.zeros_like(phi))
        if kind == "divkgrad":
            tree = (ops["DivX"](ops["InterpC2FX"](fk) * ops["GradX"](fphi))
                    + ops["DivY"](ops["InterpC2FY"](fk) * ops["GradY"](fphi))
                    + ops["DivZ"](ops["InterpC2FZ"](fk) * ops["GradZ"](fphi)))
            return {"run": _run_assign, **_assign_state(out, tree)}
        if kind == "reduce":
            exprs = [(nh.serialize(nh.E(fphi)), _abi.RED_MAX, 1), (nh.serialize(nh.E(fphi)), _abi.RED_NORM, 0),
                     (nh.serialize(fphi * fk), _abi.RED_SUM, 1)]
            return {"run": _run_reduce, "exprs": exprs, "out": torch.zeros(3, device=DEV, dtype=F64)}
        if case["tree"] == "upwind":
            u = [_field(layout.like(loc), _wrap(v)) for loc, v in zip(("SSurfX", "SSurfY", "SSurfZ"), _faces(n, seed))]
            lo, hi = W.upwind_ops()
            fk.gpu.mul_(1e-3)
            tree = fphi + _transport_dt(n) * W.transport_rhs(ops, fphi, fk, u, lo, hi)
        elif case["tree"] == "reaction":
            tree = nh.cond(fphi > 0.0, fk * nh.exp(-1.0 * fphi))(0.0) - 0.1 * fphi
        else:
            tree = db[("Filter", "SVol", "SVol")](fphi)
        return {"run": _run_assign, **_assign_state(out, tree)}
    if kind == "diffusion_grad":
        dt, w = _diffusion_dt(n), _wrap(_waves(n, seed + 1)).reshape(-1)
        phi, k = phi.reshape(-1).requires_grad_(), k.reshape(-1).requires_grad_()
        return {"run": _run_diffusion, "args": (phi, k, layout, coefs, dt, case["steps"], case["every"]), "w": w}
    faces = [layout.like(loc) for loc in ("SSurfX", "SSurfY", "SSurfZ")]
    u = [_wrap(v).reshape(-1) for v in _faces(n, seed)]
    k = k.mul_(1e-3).reshape(-1)
    phi, dt = phi.reshape(-1), _transport_dt(n)
    if kind == "transport_step":
        return {"run": _run_transport_step, "layout": layout, "faces": faces, "phi": phi, "k": k, "u": u,
                "coefs": coefs, "dt": dt, "s": [torch.zeros_like(phi) for _ in range(3)]}
    w = _wrap(_waves(n, seed + 1)).reshape(-1)
    return {"run": _run_transport, "w": w,
            "args": (phi.requires_grad_(), k.requires_grad_(), layout, faces, u, coefs, dt, case["steps"],
                     case["every"])}


def run(state):
    return state["run"](state)


def _run_assign(st):
    _abi.check(nh.lib().nebo_assign(*st["args"], 1, _stream()))
    return st["lhs"].gpu


def _run_heat(st):
    h = st["stepper"]
    h.step(0)
    return h.fields[1].gpu, h.red


def _run_reduce(st):
    out, lib, s = st["out"], nh.lib(), _stream()
    for i, (e, op, ghosts) in enumerate(st["exprs"]):
        _abi.check(lib.nebo_reduce_async(e.ref, op, ghosts, C.c_void_p(out.data_ptr() + 8 * i), s))
    return out


def _run_batch(st):
    st["batch"].step(0)
    return st["out"]


def _run_diffusion(st):
    phi, k = st["args"][:2]
    end = adjoint.DiffusionTrajectory.apply(*st["args"])
    return (end.detach(), *torch.autograd.grad(end, (phi, k), st["w"]))


def _run_transport_step(st):
    a, (s1, s2, out) = st, st["s"]
    rest = (a["k"], a["u"], a["coefs"], a["dt"])
    transport.stage(a["layout"], s1, a["phi"], None, *rest, 1, a["faces"])
    transport.stage(a["layout"], s2, a["phi"], s1, *rest, 2, a["faces"])
    transport.stage(a["layout"], out, a["phi"], s2, *rest, 3, a["faces"])
    return out


def _run_transport(st):
    phi, k = st["args"][:2]
    end = transport.TransportTrajectory.apply(*st["args"])
    return (end.detach(), *torch.autograd.grad(end, (phi, k), st["w"]))


def _run_p2c(st):
    return st["op"].apply_to_field(st["src"], st["dest"]).gpu


def _run_c2p(st):
    return st["op"].apply_to_field(st["src"], st["dest"])


# ---- what a pass cannot do without ------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "batch":
        dims = _dims(case)
        blocks = sum((d[0] + 2) * (d[1] + 2) * (d[2] + 2) for d in dims)
        cells = sum(d[0] * d[1] * d[2] for d in dims)
        return {"bytes": 8 * (blocks + cells), "flops": 23 * cells}
    if kind == "heat":
        cells = case["n"] ** 3
        return {"bytes": 16 * (case["n"] + 2) ** 3, "flops": 25 * cells}
    n = _n(case)
    cells = n[0] * n[1] * n[2]
    if kind in ("p2c", "c2p"):
        m = case["particles"]   # an edge of 0.85 cells overlaps 1.85^3 cells on average
        return {"bytes": 40 * m + 8 * cells, "flops": 6.3 * 12 * m}
    if kind == "divkgrad":
        return {"bytes": 24 * cells, "flops": 48 * cells}
    if kind == "reduce":   # the three results come from two fields
        return {"bytes": 16 * cells, "flops": 5 * cells}
    if kind == "expr":
        fields, flops = {"upwind": (6, 80), "reaction": (3, 25), "filter": (2, 28)}[case["tree"]]
        return {"bytes": 8 * fields * cells, "flops": flops * cells}
    if kind == "diffusion_grad":   # each state is a whole field: steps read and write theirs
        s, e = case["steps"], case["every"]
        return {"bytes": cells * (24 * s + 24 * (s - s // e) + 48 * s), "flops": cells * (48 * s + 48 * (s - s // e) + 100 * s)}
    stage = (48 + 56 + 56) * cells
    if kind == "transport_step":
        return {"bytes": stage, "flops": 3 * 85 * cells}
    s = case["steps"]
    return {"bytes": s * (2 * stage + (80 + 88 + 80) * cells), "flops": s * cells * (6 * 85 + 3 * 150)}


# ---- the same in plain torch, 64 bits ----------------------------------------


def _along(a, axis, by):
    return torch.roll(a, by, axis)   # by = 1: each place gets the value below it


def _diffusion(phi, k, n):
    """div(interp(k) grad(phi)) of a periodic interior (z, y, x), unit edges."""
    out = 0.0
    for axis, m in ((2, n[0]), (1, n[1]), (0, n[2])):
        f = 0.5 * (_along(k, axis, 1) + k) * ((phi - _along(phi, axis, 1)) * m)
        out = out + (_along(f, axis, -1) - f) * m
    return out


def _transport_rhs(phi, k, u, n):
    out = _diffusion(phi, k, n)
    for (axis, m), v in zip(((2, n[0]), (1, n[1]), (0, n[2])), u):
        f = torch.where(v > 0.0, _along(phi, axis, 1), phi) * v
        out = out - (_along(f, axis, -1) - f) * m
    return out


def _rk3(phi, k, u, n, dt):
    s1 = phi + dt * _transport_rhs(phi, k, u, n)
    s2 = 0.75 * phi + 0.25 * (s1 + dt * _transport_rhs(s1, k, u, n))
    return phi / 3.0 + (2.0 / 3.0) * (s2 + dt * _transport_rhs(s2, k, u, n))


def _pad(a):
    return torch.nn.functional.pad(a, (1, 1, 1, 1, 1, 1)).reshape(-1)


def _laplacian_euler(block, n, s):
    """phi + s*lapl(phi) of the interior of a ghosted block."""
    c = block[1:-1, 1:-1, 1:-1]
    lap = ((block[1:-1, 1:-1, 2:] - 2 * c + block[1:-1, 1:-1, :-2]) * n[0] ** 2
           + (block[1:-1, 2:, 1:-1] - 2 * c + block[1:-1, :-2, 1:-1]) * n[1] ** 2
           + (block[2:, 1:-1, 1:-1] - 2 * c + block[:-2, 1:-1, 1:-1]) * n[2] ** 2)
    return c + s * lap


def exact(case, seed):
    kind = case["kind"]
    if kind == "heat":
        m = case["n"]
        new = _laplacian_euler(_heat_start(m, seed), (m, m, m), 0.1 / m ** 2)
        return _pad(new), torch.stack([_pad(new).max(), new.sum()])
    if kind == "batch":
        dims = _dims(case)
        at, total = _starts(dims)
        a, b = _rand(_gen(seed), total, -1.0, 1.0), torch.zeros(total, device=DEV, dtype=F64)
        for o, d in zip(at, dims):
            shape = (d[2] + 2, d[1] + 2, d[0] + 2)
            cut = slice(o, o + shape[0] * shape[1] * shape[2])
            b[cut].view(shape)[1:-1, 1:-1, 1:-1] = _laplacian_euler(a[cut].view(shape), (1, 1, 1), 0.1)
        return b
    n = _n(case)
    if kind in ("p2c", "c2p"):
        pos, size, vals = _particles(case, seed)
        lo = [p - size * 0.5 for p in pos]
        first = [torch.floor(v).long() for v in lo]
        # window cells carry one ghost layer, which no particle here overlaps
        X, Y = n[0] + 2, n[1] + 2
        cells = torch.zeros(X * Y * (n[2] + 2), device=DEV, dtype=F64) if kind == "p2c" else _wrap(_waves(n, seed)).reshape(-1)
        got = torch.zeros_like(vals)
        for dz in range(3):
            for dy in range(3):
                for dx in range(3):
                    share, at = torch.ones_like(vals), []
                    for a, d in enumerate((dx, dy, dz)):
                        i = first[a] + d
                        share = share * torch.clamp(torch.minimum(i + 1.0, lo[a] + size) - torch.maximum(i.double(), lo[a]), min=0.0) / size
                        at.append(torch.clamp(i, max=n[a]) + 1)
                    flat = at[0] + X * (at[1] + Y * at[2])
                    if kind == "p2c":
                        cells.index_add_(0, flat, share * vals)
                    else:
                        got += share * cells[flat]
        return cells if kind == "p2c" else got
    phi, k = _waves(n, seed), _coef(n, seed)
    if kind == "divkgrad":
        return _pad(_diffusion(phi, k, n))
    if kind == "reduce":
        p, q = _wrap(phi), _wrap(k)
        return torch.stack([p.max(), phi.square().sum().sqrt(), (p * q).sum()])
    if kind == "expr":
        if case["tree"] == "upwind":
            return _pad(phi + _transport_dt(n) * _transport_rhs(phi, 1e-3 * k, _faces(n, seed), n))
        if case["tree"] == "reaction":
            p = _wrap(phi)
            return (torch.where(p > 0.0, _wrap(k) * torch.exp(-p), 0.0) - 0.1 * p).reshape(-1)
        s = sum(_along(_along(_along(phi, 0, a), 1, b), 2, c) for a in (1, 0, -1) for b in (1, 0, -1) for c in (1, 0, -1))
        return _pad(s / 27.0)
    if kind == "transport_step":
        return _wrap(_rk3(phi, 1e-3 * k, _faces(n, seed), n, _transport_dt(n))).reshape(-1)
    phi.requires_grad_()
    k = (k if kind == "diffusion_grad" else 1e-3 * k).requires_grad_()
    end = phi
    for _ in range(case["steps"]):
        if kind == "diffusion_grad":
            end = end + _diffusion_dt(n) * _diffusion(end, k, n)
        else:
            end = _rk3(end, k, _faces(n, seed), n, _transport_dt(n))
    gphi, gk = torch.autograd.grad(end, (phi, k), _waves(n, seed + 1))
    return _wrap(end.detach()).reshape(-1), _wrap(gphi).reshape(-1), _pad(gk)


__all__ = ["listed", "draw", "prepare", "run", "work", "exact"]
