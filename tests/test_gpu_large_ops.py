"""Eager ops above 330 MB on rows of whole cache lines, where they leave the caches alone, and D3Q27 steps with a mask
and a boundary over both kinds of store.

Ops act on each cell, or each plane, alone: the halves of a large state, which lie below that line, are their
reference.  A small periodic grid repeated along z is the reference of a large one.  The kernels differ in loads,
stores and order alone; the bar is the one between two kernels of the same update, 4 ulp everywhere and 99.9 %
identical; what only moves values is exact."""

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


def _large(q, shape, dtype):
    g = torch.Generator("cuda:0").manual_seed(sum(shape))
    w = torch.from_numpy(F.LATS[q].w).to("cuda:0", dtype).reshape((-1,) + (1,) * len(shape))
    return w * (1 + 0.05 * torch.rand((q,) + shape, device="cuda:0", dtype=dtype, generator=g))


CASES = [
    (19, (68, 128, 256), torch.float64, ("collide_bgk3d", "collide_mrt3d"), "stream3d", "macroscopic3d"),
    (19, (141, 250, 128), torch.float32, ("collide_bgk3d", "collide_cascaded_d3q19"), "stream3d", "macroscopic3d"),
    (27, (64, 99, 544), torch.float32, ("collide_bgk27", "collide_cumulant_geier_d3q27"), "stream27", "macroscopic27"),
    (9, (3102, 3104), torch.float32, ("collide_bgk", "collide_mrt"), "stream", "macroscopic"),
]


@pytest.mark.parametrize("q,shape,dtype,collide,stream,macro", CASES)
def test_ops_on_halves(q, shape, dtype, collide, stream, macro):
    f = _large(q, shape, dtype)
    mb = f.numel() * f.element_size() / 1e6
    assert mb > 330 > mb / 2 and shape[-1] * f.element_size() % 128 == 0
    h = shape[0] // 2
    halves = [f[:, :h].contiguous(), f[:, h:].contiguous()]
    for name in collide:
        op = getattr(tl, name)
        _same(op(f, 0.7), torch.cat([op(v, 0.7) for v in halves], 1))
    m = getattr(tl, macro)
    for whole, a, b in zip(m(f), *[m(v) for v in halves]):
        assert torch.equal(whole, torch.cat([a, b]))
    g = getattr(tl, stream)(f)
    c = F.LATS[q].c
    axes = tuple(range(len(shape)))
    for k in range(q):
        shift = tuple(int(v) for v in c[k][:len(shape)][::-1])
        assert torch.equal(g[k], torch.roll(f[k], shift, axes))


@pytest.mark.parametrize("shape,dtype", [c[1:3] for c in CASES[:2]])
def test_boundary_op_on_halves(shape, dtype):
    f = _large(19, shape, dtype)
    h = shape[0] // 2
    wall = torch.zeros(shape, dtype=torch.bool, device="cuda:0")
    wall[:, 0] = wall[:, -1] = True
    body = torch.zeros_like(wall)
    body[:, 3:6, 4:9] = True
    cut = lambda v: (v[:h].contiguous(), v[h:].contiguous())
    bc = lambda v, m, s: tl.apply_simple_channel_boundaries_3d(v, 0.04, m, s)
    parts = [bc(v.contiguous(), m, s) for v, m, s in zip((f[:, :h], f[:, h:]), cut(wall), cut(body))]
    _same(bc(f, wall, body), torch.cat(parts, 1))


# rows of 106, 212 and 424 bytes (partial sectors) and of 64 cells; copies below 20 MB, for 20-145 MB and beyond
@pytest.mark.parametrize("dtype,nx,copies", [
    (torch.float16, 53, (14, 80)), (torch.float32, 53, (7, 45)), (torch.float64, 53, (4, 25)),
    (torch.float32, 64, (6, 40)), (torch.bfloat16, 50, (14, 150)),
])
@pytest.mark.parametrize("collision", ["bgk", "mrt", "cm", "cumulant", "geier"])
def test_repeated_d3q27_channels(collision, dtype, nx, copies):
    shape = (10, 67, nx)
    dev_store = dtype in (torch.float16, torch.bfloat16)
    f = F.random_state(27, shape, seed=nx, noise=2e-3, u_amp=0.03)
    if dev_store:
        f = f - F.LATS[27].w.reshape(-1, 1, 1, 1)
    f = torch.from_numpy(f).to("cuda:0", dtype)
    solid = torch.zeros(shape, dtype=torch.int8, device="cuda:0")
    solid[5, 33:, 3:9] = 1
    kw = dict(lattice="D3Q27", collision=collision, deviation=dev_store, boundary="channel_x", u_bc=(0.04, 0.0, 0.0),
              temporal_blocking=False)
    if collision == "geier":
        kw["rates"] = (1.1, 1.0, 0.9)
    ref = tl.FusedSolver3D(*shape, 0.6, "cuda:0", dtype, solid=solid, **kw).run(f, 3)[0].clone()
    for k in copies:
        big = tl.FusedSolver3D(shape[0] * k, *shape[1:], 0.6, "cuda:0", dtype, solid=solid.repeat(k, 1, 1), **kw)
        g = big.run(f.repeat(1, k, 1, 1), 3)[0]
        for i in (0, k // 2, k - 1):
            _same(ref, g[:, 10 * i:10 * (i + 1)])


# planes whose last piece of 8192 values is whole, a few groups, or ends inside a group
@pytest.mark.parametrize("ny,nx", [(64, 128), (64, 129), (91, 91), (3, 5), (127, 130)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
def test_mass_correction_of_planes(ny, nx, dtype):
    f = (0.02 + torch.rand((19, 5, ny, nx), generator=torch.Generator().manual_seed(nx))).to(dtype).to("cuda:0")
    big = torch.zeros((19, 7, ny, nx), dtype=dtype, device="cuda:0")
    big[:, 1:-1] = f
    total = float(f.double().sum())
    tl.apply_mass_correction(big[:, 1:-1], 0.9 * total)
    want, eps = f.double() * 0.9, torch.finfo(dtype).eps  # one rounding of the scale, one of the product
    assert bool(((big[:, 1:-1].double() - want).abs() <= 2 * eps * want).all())
    assert not big[:, 0].any() and not big[:, -1].any()
