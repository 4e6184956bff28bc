"""run() as one library call: the same launches, buffers and results as step() / step2() in a loop."""

from __future__ import annotations

import pytest
import torch

import tensorlbm_amd as tl
from tests import _fields as F

pytestmark = pytest.mark.gpu


def _solver(dtype, closure=None, **kw):
    dev = dtype == torch.float16
    return tl.FusedSolver3D(5, 7, 21, 0.6, "cuda:0", dtype, deviation=dev, closure=closure, **kw)


def _start(dtype):
    f = F.random_state(19, (5, 7, 21), seed=2, noise=2e-3, u_amp=0.03)
    if dtype == torch.float16:
        f = f - F.LATS[19].w.reshape(-1, 1, 1, 1)
    return torch.from_numpy(f).to("cuda:0", dtype)


@pytest.mark.parametrize("n", [0, 1, 2, 3, 8, 1027])
@pytest.mark.parametrize("dtype,two", [(torch.float32, True), (torch.float32, False), (torch.float64, False),
                                       (torch.float16, True), (torch.float16, False)])
def test_run_equals_steps(n, dtype, two):
    a, b = (_solver(dtype, temporal_blocking=two) for _ in range(2))
    f0 = _start(dtype)
    kept = f0.clone()
    f, diags = a.run(f0, n)
    g = f0
    for _ in range(n // 2 if b.two_step else n):
        g = b.step2(g) if b.two_step else b.step(g)
    if b.two_step and n % 2:
        g = b.step(g)
    assert len(diags) == n and torch.equal(f, g) and torch.equal(f0, kept)
    assert (f is f0) if n == 0 else f.data_ptr() in (a._buf_a.data_ptr(), a._buf_b.data_ptr())
    if n:  # continuing from a buffer never writes into it before it is read
        h, _ = a.run(f, 3)
        g, _ = b.run(g, 3)
        assert torch.equal(h, g)


def test_run_with_closure_sees_updated_weights():
    m = tl.EddyViscosityMLP3D("cuda:0", seed=1)
    s, t = (_solver(torch.float16, closure=m) for _ in range(2))
    f0 = _start(torch.float16)
    s.run(f0, 2)
    m.params[:m.nparam] *= 3.0
    m.mark_updated()
    f, _ = s.run(f0, 2)
    assert torch.equal(f, t.step(t.step(f0)))


def test_run_uses_an_overridden_step():
    class Counting(tl.FusedSolver3D):
        calls = 0

        def step(self, f, **kw):
            Counting.calls += 1
            return super().step(f, **kw)

    s = Counting(4, 4, 8, 0.6, "cuda:0", torch.float64)
    s.run(torch.rand(19, 4, 4, 8, dtype=torch.float64, device="cuda:0"), 5)
    assert Counting.calls == 5


def test_run_refuses_bad_input():
    s = _solver(torch.float32)
    with pytest.raises(ValueError, match="dtype"):
        s.run(_start(torch.float64), 4)
    with pytest.raises(ValueError, match="shape"):
        s.run(torch.zeros(19, 5, 7, 20, device="cuda:0"), 4)


@pytest.mark.parametrize("dtype,deviation", [(torch.float32, False), (torch.float64, False), (torch.float16, True),
                                             (torch.bfloat16, True), (torch.float16, False)])
def test_cavity_fill(dtype, deviation):
    b = tl.BatchedCavities([3, 5, 64, 33], [0.7] * 4, dtype=dtype, deviation=deviation)
    b.a.fill_(7.0)
    b.fill_equilibrium()
    w = tl.lattice.D3Q19.W_EXACT64.to("cuda:0").to(dtype)
    for i in range(4):
        want = torch.zeros_like(w) if deviation else w
        assert torch.equal(b.cavity(i), want.reshape(19, 1, 1, 1).expand_as(b.cavity(i)))
        b.cavity(i).fill_(7.0)
    assert bool((b.a == 7.0).all())  # the padding is not written
