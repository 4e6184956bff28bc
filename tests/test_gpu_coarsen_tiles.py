"""Block averages at the edges of their launch shapes: factor 1, factors that do and do not divide a wave,
one coarse cell per workgroup and factors beyond its 512 lanes, odd rows, against float64 block means."""

from __future__ import annotations

import pytest
import torch

from tensorlbm_amd import closure as cl
from tensorlbm_amd.fused import padded_populations
from tests import _fields as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,r", [((3, 4, 5), 1), ((2, 4, 6), 2), ((3, 6, 129), 3), ((6, 3, 768), 3), ((4, 8, 516), 4),
                                     ((5, 5, 35), 5), ((7, 7, 7), 7), ((64, 64, 64), 64), ((2, 2, 1026), 2)])
@pytest.mark.parametrize("dtype,deviation", [(torch.float32, False), (torch.float64, False), (torch.float16, True)])
@pytest.mark.parametrize("padded", [False, True])
def test_coarsen_shapes(shape, r, dtype, deviation, padded):
    nz, ny, nx = shape
    f = torch.from_numpy(F.random_state(19, shape, seed=nx + r, noise=2e-3, u_amp=0.04))
    w = torch.from_numpy(F.LATS[19].w).reshape(-1, 1, 1, 1)
    c = torch.from_numpy(F.LATS[19].c).double()
    stored = ((f - w) if deviation else f).to(dtype)
    f = stored.double() + (w if deviation else 0)
    dev = stored.to("cuda:0")
    if padded:
        buf = padded_populations(19, nz, ny, nx, dtype, "cuda:0")
        buf.copy_(dev)
        dev = buf
    got = cl.coarsen_moments(dev, r, deviation=deviation).double().cpu()
    rho = f.sum(0)
    u = torch.einsum("qd,qzyx->dzyx", c, f) / rho
    fields = [rho, *u, u[0] ** 2, u[1] ** 2, u[2] ** 2, u[0] * u[1], u[0] * u[2], u[1] * u[2]]
    want = torch.stack([v.reshape(nz // r, r, ny // r, r, nx // r, r).mean((1, 3, 5)) for v in fields])
    # per-cell moments in fp32 (19 terms of at most 1/3): ~1e-6 on rho and u, twice that on products with u < 0.2
    assert got.shape == want.shape
    assert float((got - want).abs().max()) <= 2e-6
