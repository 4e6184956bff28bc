"""Block averages with factors beyond the 512 lanes of a workgroup (and at that line), where the lanes of the one
coarse cell walk along its row, against float64 block means."""

from __future__ import annotations

import pytest
import torch

from tensorlbm_amd import closure as cl
from tests import _fields as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r,cells", [(511, 2), (512, 2), (513, 2), (600, 1)])
@pytest.mark.parametrize("dtype,deviation", [(torch.float32, False), (torch.float64, False), (torch.float16, True)])
def test_factors_beyond_the_lanes(r, cells, dtype, deviation):
    nx = r * cells
    f = torch.from_numpy(F.random_state(19, (1, 1, nx), seed=r, noise=2e-3, u_amp=0.04))
    w = torch.from_numpy(F.LATS[19].w).reshape(-1, 1, 1, 1)
    c = torch.from_numpy(F.LATS[19].c).double()
    stored = ((f - w) if deviation else f).to(dtype)
    f = stored.double() + (w if deviation else 0)
    # r x r rows that all lie in one place: the operator takes its strides from the tensor
    got = cl.coarsen_moments(stored.to("cuda:0").expand(19, r, r, nx), r, deviation=deviation).double().cpu()
    rho = f.sum(0)
    u = torch.einsum("qd,qzyx->dzyx", c, f) / rho
    fields = [rho, *u, u[0] ** 2, u[1] ** 2, u[2] ** 2, u[0] * u[1], u[0] * u[2], u[1] * u[2]]
    want = torch.stack([v.reshape(1, 1, cells, r).mean(3) for v in fields])
    # per-cell moments in fp32 (19 terms of at most 1/3): ~1e-6 on rho and u, twice that on products with u < 0.2
    assert got.shape == want.shape == (10, 1, 1, cells)
    assert float((got - want).abs().max()) <= 2e-6
