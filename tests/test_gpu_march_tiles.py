"""The z march of the two-step launch at each of its tile shapes and kinds of store, on grids above the small-grid
line, where the march and not the block kernel runs (test_gpu_tiles.py has the same rows on grids below it).

The line is 800 cells per compute unit; every grid here is given enough planes to lie above it on the device at
hand.  The bar is the one between the two kernels: 4 ulp of the stored type everywhere, 99.9 % identical; the integer
canary is exact."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import tensorlbm_amd as tl
from oracle import ref
from tests import _fields as F

pytestmark = pytest.mark.gpu

ULP = {torch.float32: 2.0**-23, torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7}
ROWS = [
    (3, 16), (23, 17), (50, 32), (23, 48), (37, 63), (31, 96), (31, 108),  # full rows
    (19, 109), (9, 128),  # base tile
    (17, 131), (29, 211), (11, 255),  # wide parts
]


def _planes(ny, nx, odd=3):
    """Planes enough to lie above the small-grid line."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nz = 800 * cus // (ny * nx) + odd
    assert nz * ny * nx > 800 * cus
    return nz


def _state(shape, dtype, deviation, seed):
    g = torch.Generator("cuda:0").manual_seed(seed)
    fields = [torch.randn(shape, device="cuda:0", generator=g, dtype=torch.float64) for _ in range(4)]
    f = tl.equilibrium3d(1 + 0.02 * fields[0], *(0.03 * u for u in fields[1:]))
    w = torch.from_numpy(F.LATS[19].w).to("cuda:0").reshape(-1, 1, 1, 1)
    f += 2e-3 * w * torch.randn(f.shape, device="cuda:0", generator=g, dtype=torch.float64)
    return (f - w if deviation else f).to(dtype)


def _pair(shape, dtype, boundary, collision="bgk", layout="padded"):
    nz, ny, nx = shape
    deviation = dtype != torch.float32
    f = _state(shape, dtype, deviation, nx + ny)
    solid = torch.zeros(shape, dtype=torch.int8, device="cuda:0")
    solid[nz // 2 - 1:nz // 2 + 2, ny // 2, 2:max(3, nx // 2)] = 1
    kw = dict(deviation=deviation, solid=solid if boundary else None, boundary=boundary, u_bc=(0.04, 0.0, 0.0),
              collision=collision, layout=layout)
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


@pytest.mark.parametrize("ny,nx", ROWS)
@pytest.mark.parametrize("dtype,boundary", [(torch.float32, "channel_x"), (torch.float32, None),
                                            (torch.float32, "lid_y"), (torch.float16, "far_field"),
                                            (torch.bfloat16, "channel_x")])
def test_marched_tiles_match_single_steps(ny, nx, dtype, boundary):
    _same(*_pair((_planes(ny, nx), ny, nx), dtype, boundary))


@pytest.mark.parametrize("ny,nx", [(37, 63), (19, 109), (29, 211)])
@pytest.mark.parametrize("collision", ["mrt", "cm", "cumulant"])
@pytest.mark.parametrize("layout", ["padded", "contiguous"])
def test_marched_collisions_match_single_steps(ny, nx, collision, layout):
    _same(*_pair((_planes(ny, nx), ny, nx), torch.float32, "channel_x", collision, layout))


@pytest.mark.parametrize("ny,nx", [(3, 4), (7, 1), (1, 9), (1, 130), (2, 2)])
def test_marched_grids_smaller_than_a_tile(ny, nx):
    _same(*_pair((_planes(ny, nx), ny, nx), torch.float32, None))


# rows of partial lines by the size of one lattice (76 bytes a cell): 45-120 MB through L2, 120-256 MB past it,
# larger ones through L2 again
@pytest.mark.parametrize("shape", [(80, 80, 117), (95, 90, 131), (100, 100, 100), (120, 130, 117), (120, 130, 141),
                                   (150, 160, 150)])
@pytest.mark.parametrize("boundary", ["channel_x", None])
def test_kinds_of_store_match_single_steps(shape, boundary):
    _same(*_pair(shape, torch.float32, boundary))


@pytest.mark.parametrize("ny,nx", [(23, 17), (37, 62), (19, 109), (17, 131)])
def test_canary_addressing_of_the_march(ny, nx):
    nz = _planes(ny, nx, odd=1)
    solid = ref.sphere_mask(nx, ny, nz, 8.0, 8.0, nz // 2, 4.5)
    fc = np.arange(19.0 * nz * ny * nx).reshape(19, nz, ny, nx)  # every value once
    assert fc.max() < 2**23  # exact in fp32, with room for the 1e-9 that the collision moves them by
    two = tl.FusedSolver3D(nz, ny, nx, 1e9, "cuda:0", torch.float32, solid=torch.from_numpy(solid))
    assert two.two_step
    got = two.step2(torch.from_numpy(fc).to("cuda:0", torch.float32)).cpu().numpy()
    want = ref.fullway_pull(ref.fullway_pull(fc, solid), solid)
    assert int((got.round().astype(np.int64) != want.round().astype(np.int64)).sum()) == 0
