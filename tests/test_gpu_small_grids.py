"""The two-step launch on either side of its small-grid line, against one-step launches.

Grids of at most 800 cells per compute unit (204 800 cells on 256) take the block kernel, larger
ones the z march.  The blocks here are cut from whole axes and from remainders of one cell, wrap in
one, two or all three axes, and include axes of one cell; the marched grids lie just above the line.
The bar is the one between the two kernels: 4 ulp of the stored type everywhere, 99.9 % identical.
"""

from __future__ import annotations

import pytest
import torch

import tensorlbm_amd as tl
from tests import _fields as F

pytestmark = pytest.mark.gpu

ULP = {torch.float32: 2.0**-23, torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7}
BLOCKS = [
    (1, 1, 4), (1, 1, 2000), (1, 900, 5), (300, 1, 7), (2, 3, 4), (3, 2, 130), (8, 8, 8), (13, 17, 19), (24, 24, 48),
    (31, 29, 45), (64, 50, 64), (61, 53, 63),
]
MARCHED = [(70, 30, 100), (130, 50, 32), (30, 66, 109), (25, 64, 131), (20, 50, 211)]


def _pair(shape, dtype, boundary, collision="bgk", **extra):
    nz, ny, nx = shape
    dev_store = dtype != torch.float32
    f = F.random_state(19, shape, seed=nx + ny, noise=2e-3, u_amp=0.03)
    if dev_store:
        f = f - F.LATS[19].w.reshape(-1, 1, 1, 1)
    f = torch.from_numpy(f).to("cuda:0", dtype)
    solid = torch.zeros(shape, dtype=torch.int8, device="cuda:0")
    solid[nz // 2, ny // 2, 2:max(3, nx // 2)] = 1
    kw = dict(deviation=dev_store, solid=solid if boundary else None, boundary=boundary, u_bc=(0.04, 0.0, 0.0),
              collision=collision, **extra)
    one = tl.FusedSolver3D(nz, ny, nx, 0.6, "cuda:0", dtype, temporal_blocking=False, **kw)
    two = tl.FusedSolver3D(nz, ny, nx, 0.6, "cuda:0", dtype, temporal_blocking=True, **kw)
    if not two.two_step:
        pytest.skip("the outlet column rules two-step launches out on this grid")
    a = b = f
    for _ in range(2):
        a = one.step(one.step(a))
        b = two.step2(b)
    return a, b


def _same(a, b):
    x, y = a.double(), b.double()
    assert torch.isfinite(x).all()
    diff = (x - y).abs()
    assert bool((diff <= 4 * ULP[a.dtype] * torch.maximum(x.abs(), y.abs()) + 1e-30).all())
    assert float((diff == 0).double().mean()) >= 0.999


@pytest.mark.parametrize("shape", BLOCKS + MARCHED)
@pytest.mark.parametrize("dtype,boundary", [(torch.float32, "channel_x"), (torch.float32, None), (torch.float32, "lid_y"),
                                            (torch.float16, "far_field"), (torch.bfloat16, "channel_x")])
def test_either_side_matches_single_steps(shape, dtype, boundary):
    _same(*_pair(shape, dtype, boundary))


@pytest.mark.parametrize("shape", [(13, 17, 19), (70, 30, 100)])
@pytest.mark.parametrize("collision", ["mrt", "cm", "cumulant"])
@pytest.mark.parametrize("layout", ["padded", "contiguous"])
def test_collisions_match_single_steps(shape, collision, layout):
    _same(*_pair(shape, torch.float32, "channel_x", collision, layout=layout))
