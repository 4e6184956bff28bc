"""The two-step launch over grids that take each of its tile shapes, against one-step launches.

The tile follows the grid (full rows up to 108 cells, the row in equal parts wider than 64 from
129, else 64 x 8) and so does the way results are stored; the per-cell code does not, so the bar is
the one between the two kernels: 4 ulp of the stored type everywhere, 99.9 % of values identical.
"""

from __future__ import annotations

import pytest
import torch

import tensorlbm_amd as tl
from tests import _fields as F

pytestmark = pytest.mark.gpu

ULP = {torch.float32: 2.0**-23, torch.float16: 2.0**-10}
SHAPES = [
    (70, 3, 16), (9, 23, 17), (40, 50, 32), (9, 23, 48), (5, 37, 63), (7, 31, 96), (7, 31, 108),  # full rows
    (6, 19, 109), (5, 9, 128),  # base tile
    (5, 17, 131), (4, 29, 211), (3, 11, 255),  # wide parts
]


def _same(a, b):
    x, y = a.double(), b.double()
    assert torch.isfinite(x).all()
    diff = (x - y).abs()
    assert bool((diff <= 4 * ULP[a.dtype] * torch.maximum(x.abs(), y.abs()) + 1e-30).all())
    assert float((diff == 0).double().mean()) >= 0.999


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype,boundary", [(torch.float32, "channel_x"), (torch.float32, None),
                                            (torch.float16, "far_field")])
@pytest.mark.parametrize("layout", ["padded", "contiguous"])
def test_tile_shapes_match_single_steps(shape, dtype, boundary, layout):
    nz, ny, nx = shape
    dev_store = dtype == torch.float16
    f = F.random_state(19, shape, seed=nx, noise=2e-3, u_amp=0.03)
    if dev_store:
        f = f - F.LATS[19].w.reshape(-1, 1, 1, 1)
    f = torch.from_numpy(f).to("cuda:0", dtype)
    solid = torch.zeros(shape, dtype=torch.int8, device="cuda:0")
    solid[nz // 2, ny // 2, 2:nx // 2] = 1
    kw = dict(deviation=dev_store, solid=solid if boundary else None, boundary=boundary, u_bc=(0.04, 0.0, 0.0),
              layout=layout)
    one = tl.FusedSolver3D(nz, ny, nx, 0.6, "cuda:0", dtype, temporal_blocking=False, **kw)
    two = tl.FusedSolver3D(nz, ny, nx, 0.6, "cuda:0", dtype, temporal_blocking=True, **kw)
    assert two.two_step == (boundary is None or (nx - 1) % 64 >= 2)
    a = b = f
    for _ in range(2):
        a = one.step(one.step(a))
        b = two.step2(b)
    _same(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_cavity_tiles_match_single_steps(dtype):
    edges = [3, 5, 16, 31, 64, 100, 108, 109, 128, 129, 140]
    taus = [0.7] * len(edges)
    dev_store = dtype == torch.float16
    bs = []
    for two in (False, True):
        b = tl.BatchedCavities(edges, taus, u_lid=0.08, dtype=dtype, deviation=dev_store, temporal_blocking=two)
        b.fill_equilibrium()
        b.run(6, graph=False)
        bs.append(b)
    for i in range(len(edges)):
        x, y = bs[0].cavity(i).double(), bs[1].cavity(i).double()
        # six steps of two kernels: an ulp of the stored type per step on values up to 1/3 (f) or 0.02 (f - w)
        bound = 6 * ULP[dtype] * (1 / 3 if dtype == torch.float32 else 0.02)
        assert float((x - y).abs().max()) <= bound, edges[i]
