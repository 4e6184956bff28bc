"""The one-step kernel on tiles of consecutive cells (rows that do not fill their waves): streaming bit for bit,
collisions and the obstacle step with its force against the oracle, over rows around the wave and tile sizes."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import tensorlbm_amd as tl
from oracle import ref
from tests import _fields as F

pytestmark = pytest.mark.gpu

SHAPES = [(3, 4, 2), (2, 5, 3), (4, 3, 63), (3, 6, 65), (2, 3, 127), (2, 9, 129), (3, 5, 193), (2, 2, 300), (2, 131, 48)]


@pytest.mark.parametrize("q", [9, 19, 27])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16])
def test_stream_is_exact(q, shape, dtype):
    lat = F.LATS[q]
    dims = shape[1:] if q == 9 else shape
    f = torch.randn((q,) + dims, generator=torch.Generator().manual_seed(q + shape[2])).to(dtype).to("cuda:0")
    got = {9: tl.stream, 19: tl.stream3d, 27: tl.stream27}[q](f)
    for i, c in enumerate(np.asarray(lat.c).tolist()):
        want = torch.roll(f[i], (c[1], c[0]) if q == 9 else (c[2], c[1], c[0]), tuple(range(len(dims))))
        assert torch.equal(got[i], want), i


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("collision", ["BGK", "CM", "CUMULANT"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_obstacle_step_with_force(shape, collision, dtype):
    f = F.random_state(19, shape, seed=shape[2], noise=2e-3, u_amp=0.04)
    f = f.astype(np.float32).astype(np.float64) if dtype == torch.float32 else f.astype(np.float64)
    solid = np.random.default_rng(shape[1]).random(shape) < 0.2
    acc = torch.zeros(3, dtype=torch.float64, device="cuda:0")
    got = tl.fused_obstacle_step(torch.from_numpy(f).to("cuda:0", dtype), 0.02,
                                 torch.from_numpy(solid.astype(np.int8)).to("cuda:0"), 0.1, 1.0, collision=collision,
                                 force=acc)
    want, force = ref.fused_obstacle_step(f, 3 * 0.02 + 0.5, solid, collision=collision, cs_delta_sq=0.01,
                                          with_force=True)
    tol = 1e-6 if dtype == torch.float32 else 1e-13  # the obstacle step's bar elsewhere
    assert np.abs(got.double().cpu().numpy() - want).max() <= tol
    assert np.abs(acc.cpu().numpy() - np.asarray(force)).max() <= 1e-9 * (1 + solid.sum())
