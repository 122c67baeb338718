"""Trajectories whose scratch passes what the cache may keep (1/32 of the memory), on
two streams in turn, against the same steps called one by one, and the memory that
is free after a trim.  Bar: the same bits."""
import pytest
import torch

import nebo_hip as nh
from nebo_hip import _abi
from nebo_hip import adjoint as adj

pytestmark = pytest.mark.gpu


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_boxes_past_the_limit():
    total = torch.cuda.mem_get_info()[1]
    limit = total // 32
    # two blocks of each box as scratch: 0.16, 0.3, 0.45 and 0.62 of the limit
    sides = [round((f * limit / 16) ** (1 / 3)) for f in (0.16, 0.3, 0.45, 0.62)]
    c = nh.axis_coefs(nh.build_stencils(7, 11, 13, 1.0, 1.0, 1.0))
    dt = 1e-4
    work = []
    g = torch.Generator("cuda").manual_seed(3)
    for n in sides:
        L = nh.Layout.build((n - 2, n - 2, n - 2), 1)
        phi = torch.rand(L.npts, generator=g, device="cuda", dtype=torch.float64)
        k = torch.rand(L.npts, generator=g, device="cuda", dtype=torch.float64) + 0.5
        first, want = phi.clone(), torch.empty_like(phi)
        adj.diffusion_step(L, want, first, k, c, dt)
        adj.diffusion_step(L, first, want, k, c, dt)
        work.append((L, phi, k, first))
        del want
    _abi.call("nebo_pool_trim", 0)
    torch.cuda.empty_cache()
    start = free_bytes()
    streams = torch.cuda.Stream(), torch.cuda.Stream()
    for r in range(2):
        for i, (L, phi, k, want) in enumerate(work):
            s = streams[(i + r) % 2]
            with torch.cuda.stream(s):
                end, ckpt = adj.forward(L, phi, k, c, dt, 2, 2, stream=s)
                inside = (slice(1, -1),) * 3
                shape = L.glob[::-1]
                assert torch.equal(end.reshape(shape)[inside], want.reshape(shape)[inside])
                del end, ckpt
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    assert start - free_bytes() <= limit + (64 << 20)
    _abi.call("nebo_pool_trim", 0)
    assert start - free_bytes() <= 64 << 20
