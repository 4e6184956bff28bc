"""The one-launch companions of the obstacle step (six far-field faces, force buffers, mass correction) against
the plane writes and sums they stand for, over the layouts, types and sizes their launches distinguish."""

from __future__ import annotations

import pytest
import torch

import tensorlbm_amd as tl
from tensorlbm_amd.fused import padded_populations

pytestmark = pytest.mark.gpu

U = (0.06, 0.01, -0.02)


def _layouts(f):
    """The same values dense, in the solver's padded layout, as a slice of a larger grid, and transposed in (z, y)."""
    q, nz, ny, nx = f.shape
    yield "dense", f.clone()
    if q in (19, 27):
        p = padded_populations(q, nz, ny, nx, f.dtype, f.device)
        p.copy_(f)
        yield "padded", p
    big = torch.zeros((q, nz + 2, ny + 1, nx + 3), dtype=f.dtype, device=f.device)
    s = big[:, 1:-1, 1:, 2:-1]
    s.copy_(f)
    yield "slice", s
    t = torch.empty((q, ny, nz, nx), dtype=f.dtype, device=f.device).transpose(1, 2)
    t.copy_(f)
    yield "transposed", t


def _faces(f, face):
    """Plane by plane, as the function is written in the reference."""
    face = face[:, None, None]
    f[:, :, :, 0] = face
    if f.shape[3] >= 2:
        f[:, :, :, -1] = f[:, :, :, -2]
    f[:, :, 0, :] = face
    if f.shape[2] >= 2:
        f[:, :, -1, :] = face
    if f.shape[1] > 4:
        f[:, 0] = face
        f[:, -1] = face
    return f


@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 1, 2), (5, 2, 3), (4, 2, 1), (6, 3, 2), (7, 9, 65), (3, 70, 130)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("q", [19, 32])
def test_faces_match_plane_writes(shape, dtype, q):
    g = torch.Generator().manual_seed(q + shape[2])
    f = torch.randn((q,) + shape, generator=g).to(dtype).to("cuda:0")
    feq = torch.randn(19, generator=g, dtype=torch.float64).to("cuda:0")
    want = _faces(f.clone(), torch.cat([feq.to(dtype), torch.zeros(q - 19, dtype=dtype, device="cuda:0")]))
    for name, a in _layouts(f):
        tl.apply_far_field_bc_6face(a, *U[:1], feq_vec=feq)
        assert torch.equal(a, want), name
    one = torch.ones((1, 1, 1), dtype=torch.float64, device="cuda:0")
    e = tl.equilibrium3d(one, *(one * u for u in U))[:, 0, 0, 0]
    want = _faces(f.clone(), torch.cat([e.to(dtype), torch.zeros(q - 19, dtype=dtype, device="cuda:0")]))
    for name, a in _layouts(f):
        tl.apply_far_field_bc_6face(a, U[0], uy=U[1], uz=U[2])
        if dtype == torch.float64:  # two orders of the same double operations
            assert float((a - want).abs().max()) <= 1e-16, name
        else:
            assert torch.equal(a, want), name


@pytest.mark.parametrize("q,shape", [(19, (1, 1, 1)), (19, (3, 5, 7)), (19, (2, 33, 131)), (27, (4, 64, 64)),
                                     (19, (40, 50, 60))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16])
def test_mass_correction_over_layouts(q, shape, dtype):
    g = torch.Generator().manual_seed(q + shape[2])
    f = (0.02 + torch.rand((q,) + shape, generator=g)).to(dtype).to("cuda:0")
    total = float(f.double().sum())
    for name, a in _layouts(f):
        assert tl.apply_mass_correction(a, 0.9 * total) is a
        got, want = a.double(), f.double() * 0.9
        eps = torch.finfo(dtype).eps  # one rounding of the scale, one of the product
        assert bool(((got - want).abs() <= 2 * eps * want).all()), name
    b = f.clone()
    tl.apply_mass_correction(b, 0.9 * total)
    c = f.clone()
    tl.apply_mass_correction(c, 0.9 * total)
    assert torch.equal(b, c)  # a fixed order of summation


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16])
@pytest.mark.parametrize("shape", [(), (1,), (2,)])
def test_force_buffers(dtype, shape):
    """Added to, whatever their type and shape; one launch where they are single float32 / float64 values."""
    n = (6, 7, 9)
    f = torch.rand((19,) + n, device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(1)) * 0.05
    solid = torch.zeros(n, dtype=torch.int8, device="cuda:0")
    solid[2:4, 2:5, 3:6] = 1
    acc = torch.zeros(3, dtype=torch.float64, device="cuda:0")
    tl.fused_obstacle_step(f, 0.02, solid, 0.1, 1.0, force=acc)
    bufs = [torch.full(shape, 0.5 + i, dtype=dtype, device="cuda:0") for i in range(3)]
    tl.fused_obstacle_step(f, 0.02, solid, 0.1, 1.0, fx_buf=bufs[0], fy_buf=bufs[1], fz_buf=bufs[2])
    for i, b in enumerate(bufs):
        want = torch.full(shape, 0.5 + i, dtype=dtype, device="cuda:0") + acc[i].to(dtype)
        # the sample itself is a sum of atomics, whose order may differ from run to run in its last bits
        assert float((b - want).abs().max()) <= 4 * torch.finfo(dtype).eps * max(1.0, float(want.abs().max()))
