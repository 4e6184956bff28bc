"""One-step launches and eager ops over every kind of store and order of tiles that their size selects.

A small periodic grid repeated k times along z is the small grid's state k times over, step by
step, so the small grid (below 20 MB: non-temporal stores, first tile first) is the reference for the
large one (ordinary stores from 20 MB, runs of tiles, every second step of a run last tile first from
145 MB).  The kernels differ in their stores alone; the bar is the one between two kernels of the
same update, 4 ulp everywhere and 99.9 % identical.  Ops act on each cell, or each plane, alone: the
halves of a large state are their reference, bit for bit, and a shift along the axes that of the
stream op.
"""

from __future__ import annotations

import pytest
import torch

import tensorlbm_amd as tl
from tests import _fields as F

pytestmark = pytest.mark.gpu

ULP = {torch.float64: 2.0**-52, torch.float32: 2.0**-23, torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7}


def _same(a, b):
    x, y = a.double(), b.double()
    assert torch.isfinite(x).all()
    diff = (x - y).abs()
    assert bool((diff <= 4 * ULP[a.dtype] * torch.maximum(x.abs(), y.abs()) + 1e-30).all())
    assert float((diff == 0).double().mean()) >= 0.999


def _solid(shape):
    solid = torch.zeros(shape, dtype=torch.int8, device="cuda:0")
    solid[shape[0] // 2, shape[1] // 2:, 3:9] = 1
    return solid


def _state(q, shape, dtype):
    f = F.random_state(q, shape, seed=shape[2], noise=2e-3, u_amp=0.03)
    if dtype in (torch.float16, torch.bfloat16):
        f = f - F.LATS[q].w.reshape(-1, 1, 1, 1)
    return torch.from_numpy(f).to("cuda:0", dtype)


# rows of 106, 212, 272 and 256 bytes; copies for 20-145 MB, for 145-256 MB and beyond
@pytest.mark.parametrize("lattice,collision,dtype,boundary,nx,copies", [
    ("D3Q19", "bgk", torch.float16, "channel_x", 53, (20, 130)),
    ("D3Q19", "bgk", torch.bfloat16, "lid_y", 53, (20, 130)),
    ("D3Q19", "bgk", torch.float32, "channel_x", 53, (12, 70)),
    ("D3Q19", "bgk", torch.float64, "lid_y", 34, (12, 60, 100)),
    ("D3Q19", "bgk", torch.float32, None, 64, (12, 60)),
    ("D3Q27", "geier", torch.float16, None, 53, (14, 80)),
    ("D3Q27", "geier", torch.float32, None, 68, (6, 30, 50)),
])
def test_repeated_grids(lattice, collision, dtype, boundary, nx, copies):
    q = int(lattice[3:])
    shape = (10, 67, nx)
    f, solid = _state(q, shape, dtype), _solid(shape)
    kw = dict(lattice=lattice, collision=collision, deviation=dtype in (torch.float16, torch.bfloat16),
              boundary=boundary, u_bc=(0.04, 0.0, 0.0), temporal_blocking=False)
    small = tl.FusedSolver3D(*shape, 0.6, "cuda:0", dtype, solid=solid if boundary else None, **kw)
    ref = small.run(f, 3)[0].clone()
    for k in copies:
        big = tl.FusedSolver3D(shape[0] * k, *shape[1:], 0.6, "cuda:0", dtype,
                               solid=solid.repeat(k, 1, 1) if boundary else None, **kw)
        g = big.run(f.repeat(1, k, 1, 1), 3)[0]
        for i in (0, k // 2, k - 1):
            _same(ref, g[:, 10 * i:10 * (i + 1)])
        assert torch.equal(g[:, :10], g[:, 10 * (k - 1):])


@pytest.mark.parametrize("collision", ["BGK", "CM", "CUMULANT"])
@pytest.mark.parametrize("nx,copies", [(53, (12, 60)), (64, (12, 50))])
def test_repeated_obstacles(collision, nx, copies):
    shape = (10, 67, nx)
    f, solid = _state(19, shape, torch.float32), _solid(shape)

    def step(g, s):
        force = [torch.zeros((), dtype=torch.float64, device="cuda:0") for _ in range(3)]
        out = tl.fused_obstacle_step(g, 0.02, s, 0.1, 1.0, collision=collision, fx_buf=force[0], fy_buf=force[1],
                                     fz_buf=force[2])
        return out, torch.stack(force)

    ref, force = step(f, solid)
    for k in copies:
        g, total = step(f.repeat(1, k, 1, 1), solid.repeat(k, 1, 1))
        _same(ref, g[:, :10])
        _same(ref, g[:, -10:])
        assert bool(((total / k - force).abs() <= 1e-9 * force.abs().max()).all())


# rows of 140, 280 and 384 bytes; tiles of 64 x 4 (70, 150) and of whole rows (96)
@pytest.mark.parametrize("dtype,boundary,nx,copies", [
    (torch.float16, "channel_x", 70, (15, 90)), (torch.bfloat16, None, 150, (6, 45)),
    (torch.float32, "channel_x", 70, (8, 50)), (torch.float32, None, 150, (4, 30)), (torch.float32, "lid_y", 96, (6, 30)),
])
def test_repeated_closures(dtype, boundary, nx, copies):
    shape = (10, 67, nx)
    f, solid = _state(19, shape, dtype), _solid(shape)
    kw = dict(deviation=dtype != torch.float32, boundary=boundary, u_bc=(0.04, 0.0, 0.0), C_s=0.17,
              closure=tl.EddyViscosityMLP3D("cuda:0", seed=4))
    ref = tl.FusedSolver3D(*shape, 0.55, "cuda:0", dtype, solid=solid if boundary else None, **kw).run(f, 3)[0].clone()
    for k in copies:
        big = tl.FusedSolver3D(shape[0] * k, *shape[1:], 0.55, "cuda:0", dtype,
                               solid=solid.repeat(k, 1, 1) if boundary else None, **kw)
        g = big.run(f.repeat(1, k, 1, 1), 3)[0]
        for i in (0, k // 2, k - 1):
            _same(ref, g[:, 10 * i:10 * (i + 1)])


@pytest.mark.parametrize("dtype,shape", [(torch.float64, (101, 100, 102)), (torch.float32, (130, 128, 128)),
                                         (torch.float32, (31, 33, 35))])
def test_ops_on_halves(dtype, shape):
    f = _state(19, (1, shape[1], shape[2]), dtype).repeat(1, shape[0], 1, 1)
    f *= 1 + 1e-3 * torch.rand(f.shape, device="cuda:0", dtype=dtype)
    h = shape[0] // 2
    halves = [f[:, :h].contiguous(), f[:, h:].contiguous()]
    for op in (lambda v: tl.collide_bgk3d(v, 0.7), lambda v: tl.collide_mrt3d(v, 0.7)):
        assert torch.equal(op(f), torch.cat([op(v) for v in halves], 1))
    for whole, a, b in zip(tl.macroscopic3d(f), *[tl.macroscopic3d(v) for v in halves]):
        assert torch.equal(whole, torch.cat([a, b]))
    wall = torch.zeros(shape, dtype=torch.bool, device="cuda:0")
    wall[:, 0] = wall[:, -1] = True
    body = torch.zeros_like(wall)
    body[:, 3:6, 4:9] = True
    bc = lambda v, m, s: tl.apply_simple_channel_boundaries_3d(v, 0.04, m, s)
    whole = bc(f, wall, body)
    parts = [bc(halves[0], wall[:h].contiguous(), body[:h].contiguous()),
             bc(halves[1], wall[h:].contiguous(), body[h:].contiguous())]
    assert torch.equal(whole, torch.cat(parts, 1))
    c = F.LATS[19].c
    g = tl.stream3d(f)
    for q in range(19):
        assert torch.equal(g[q], torch.roll(f[q], (int(c[q][2]), int(c[q][1]), int(c[q][0])), (0, 1, 2)))
