"""The learned-closure march over grids that take each of its lengths (1, 2, 3 .. 16 planes), against the step in
float32 storage, which marches nothing: the stored deviations differ by their own rounding."""

from __future__ import annotations

import pytest
import torch

import tensorlbm_amd as tl
from tests import _fields as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 7), (40, 50, 65), (60, 60, 90), (61, 129, 130), (17, 800, 257),
                                   (80, 256, 200)])
@pytest.mark.parametrize("boundary", [None, "channel_x"])
def test_march_lengths(shape, boundary):
    nz, ny, nx = shape
    if boundary and nx < 4:
        pytest.skip("the channel needs an inlet, an inside and an outlet")
    f = torch.from_numpy(F.random_state(19, shape, seed=nx, noise=1e-3, u_amp=0.03).astype("float32")).to("cuda:0")
    w = torch.from_numpy(F.LATS[19].w).to("cuda:0", torch.float32).reshape(-1, 1, 1, 1)
    dev = (f - w).half()
    model = tl.EddyViscosityMLP3D("cuda:0", seed=4)
    kw = dict(closure=model, C_s=0.17, boundary=boundary, u_bc=(0.04, 0.0, 0.0))
    a = tl.FusedSolver3D(nz, ny, nx, 0.55, "cuda:0", torch.float16, deviation=True, **kw).step(dev).float()
    b = tl.FusedSolver3D(nz, ny, nx, 0.55, "cuda:0", **kw).step(dev.float() + w) - w
    # half an ulp of fp16 on deviations of at most 0.06, the fp32 sums behind them, and rare fp16 activation
    # flips of the network (below 1.5e-3 relative in nu_t, 1e-3 of the cells)
    diff = (a - b).abs()
    assert float(diff.max()) <= 1e-4
    assert float((diff > 0.06 * 2.0**-11 + 2e-7).double().mean()) <= 2e-3
