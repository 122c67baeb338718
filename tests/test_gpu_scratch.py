"""Scratch memory shared between calls, streams and threads: particle scatters and
masked assignments whose scratch differs in size, on two streams at once, before
and after the kept blocks are given back.  Bar: the oracle's bits."""
import threading

import numpy as np
import pytest
import torch

import nebo_hip as nh
from nebo_hip import _abi
from nebo_hip import particles as P
import oracle_lib as orc
from particle_cases import random_particles

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to("cuda:0")


class Scatter:
    def __init__(self, n, npart, seed):
        self.L = nh.Layout.build(n, 1, "SVol")
        src, coords, size, geom = random_particles(self.L, npart, seed)
        self.op = P.ParticleToCell(*geom)
        self.op.set_coordinate_information(*[dev(c) for c in coords], dev(size))
        self.src = dev(src)
        self.out = nh.Field.from_numpy(self.L, np.zeros(self.L.npts), where="gpu")
        want = nh.Field.from_numpy(self.L, np.zeros(self.L.npts), where="cpu")
        orc.particle_to_cell(want, src, *coords, size, geom)
        self.want = want.host

    def run(self, stream):
        self.out.gpu.fill_(3.0)
        self.op.apply_to_field(self.src, self.out, stream=stream)

    def check(self):
        assert np.array_equal(self.out.gpu.cpu().numpy(), self.want)


SETS = [((12, 9, 7), 30, 1), ((20, 17, 13), 9000, 2), ((20, 17, 13), 9500, 3), ((33, 8, 21), 40000, 4)]


def test_two_streams_share_scratch_blocks():
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    work = [Scatter(*s) for s in SETS]
    torch.cuda.synchronize()
    for _ in range(2):
        for r in range(6):
            for i, w in enumerate(work):
                s = (a, b)[(i + r) % 2]
                (a, b)[(i + r + 1) % 2].synchronize()   # the set's own buffers were last used there
                with torch.cuda.stream(s):
                    w.run(s)
        torch.cuda.synchronize()
        for w in work:
            w.check()
        _abi.call("nebo_pool_trim", 0)   # the second round starts from nothing kept


def test_threads_share_scratch_blocks():
    sets = [[Scatter(n, p, s + 10 * t) for n, p, s in SETS[:3]] for t in range(3)]
    torch.cuda.synchronize()
    errors = []

    def body(work):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for _ in range(5):
                    for w in work:
                        w.run(s)
                        s.synchronize()
                        w.check()
        except Exception as e:   # noqa: BLE001 (reported by the main thread)
            errors.append(e)

    threads = [threading.Thread(target=body, args=(w,)) for w in sets]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_masked_assignment_takes_small_blocks():
    L = nh.Layout.build((15, 11, 9), 1)
    rng = np.random.default_rng(5)
    f = nh.Field.from_numpy(L, rng.standard_normal(L.npts))
    for m in (1, 700, 3):
        pts = np.stack([rng.integers(0, e, m) for e in (15, 11, 9)], 1)
        nh.assign_points(pts, f, 2.5 * m)
        idx = (pts[:, 0] + 1) + L.glob[0] * ((pts[:, 1] + 1) + L.glob[1] * (pts[:, 2] + 1))
        f.host[idx] = 2.5 * m
    torch.cuda.synchronize()
    assert np.array_equal(f.gpu.cpu().numpy(), f.host)
