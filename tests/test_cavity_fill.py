"""The state of rest of a cavity batch: what fill_equilibrium takes and how autograd hears of it."""

from __future__ import annotations

import ctypes

import pytest
import torch

import tensorlbm_amd as tl
from tensorlbm_amd import _native as nat


@pytest.mark.parametrize("tau", [0.5, 0.3, 0.0, -1.0, float("nan")])
def test_fill_does_not_ask_for_a_stable_tau(tau):
    """The relaxation time has no part in the state of rest; the steps refuse it (host side, no GPU work)."""
    table = (nat.Cavity * 1)()
    table[0].edge, table[0].tau = 4, tau
    n = ctypes.c_int64()
    nat.check(nat.lib().tlbm_cavities_layout(table, 1, ctypes.byref(n), None), "layout")
    a, b = ctypes.c_void_p(0x1000), ctypes.c_void_p(0x2000)
    # (a capacity too small by one ends the call before a launch, after the other checks of the cavity)
    args = (n.value - 1, table, 1)
    assert nat.lib().tlbm_cavities_fill(nat.STORE_F32, a, *args, None) == nat.ERR_SHAPE
    assert b"capacity" in nat.lib().tlbm_last_error()
    assert nat.lib().tlbm_cavities_step(nat.STORE_F32, a, b, *args, 0.1, 0, None) == nat.ERR_INVALID
    assert b"tau must be" in nat.lib().tlbm_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,deviation", [(torch.float32, False), (torch.float16, True)])
def test_fill_of_cavities_that_cannot_step(dtype, deviation):
    c = tl.BatchedCavities([5, 9], [0.5, 0.7], dtype=dtype, deviation=deviation)
    c.fill_equilibrium()
    w = tl.lattice.D3Q19.W_EXACT64.to("cuda:0").reshape(19, 1, 1, 1)
    for i in range(2):
        want = (torch.zeros_like(w) if deviation else w).to(dtype).expand_as(c.cavity(i))
        assert torch.equal(c.cavity(i), want)
    with pytest.raises(ValueError, match="tau must be"):
        c.step()


class NoLibrary:
    def __getattr__(self, name):
        return lambda *a: 0


def _batch(device, monkeypatch):
    if device != "cpu":
        return tl.BatchedCavities([5], [0.7])
    c = object.__new__(tl.BatchedCavities)
    c._table = (nat.Cavity * 1)()
    c._table[0].edge, c._table[0].tau = 5, 0.7
    n = ctypes.c_int64()
    nat.check(nat.lib().tlbm_cavities_layout(c._table, 1, ctypes.byref(n), None), "layout")
    c.n, c.edges, c.device, c.dtype, c.deviation = 1, [5], torch.device("cpu"), torch.float32, False
    c._store, c.a = nat.STORE_F32, torch.zeros(n.value)
    monkeypatch.setattr(nat, "lib", lambda: NoLibrary())
    monkeypatch.setattr(nat, "stream_of", lambda t: 0)
    monkeypatch.setattr(nat, "on_current_device", lambda t: True)
    return c


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)])
def test_fill_is_a_write_to_autograd(device, monkeypatch):
    c = _batch(device, monkeypatch)
    w = torch.ones((), device=device, requires_grad=True)
    loss = (w * c.cavity(0)).sum()
    c.fill_equilibrium()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)])
def test_fill_under_a_tangent(device, monkeypatch):
    """A buffer with a tangent loses it, as under the operator the fill stands for."""
    import torch.autograd.forward_ad as fw

    c = _batch(device, monkeypatch)
    w = tl.lattice.D3Q19.W_EXACT64.to(device, torch.float32).reshape(19, 1, 1, 1)
    with fw.dual_level():
        c.a = fw.make_dual(c.a, torch.ones_like(c.a))
        c.fill_equilibrium()
        d = fw.unpack_dual(c.cavity(0))
        assert torch.equal(d.primal, w.expand_as(d.primal)) and not d.tangent.any()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,deviation", [(torch.float32, False), (torch.float64, False), (torch.float16, True),
                                             (torch.bfloat16, True)])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_fill_writes_the_cells_and_nothing_else(dtype, deviation, shift):
    """Edges whose planes are and are not whole sixteen-byte groups, buffers that do and do not start at one."""
    edges = [3, 4, 5, 8, 31, 64, 66, 91]
    c = tl.BatchedCavities(edges, [0.7] * len(edges), dtype=dtype, deviation=deviation)
    buf = torch.full((c.a.numel() + shift + 8,), 7.0, dtype=dtype, device="cuda:0")
    a = buf[shift:shift + c.a.numel()]
    nat.check(nat.lib().tlbm_cavities_fill(c._store, a.data_ptr(), a.numel(), c._table, c.n, nat.stream_of(a)), "fill")
    want = torch.full_like(buf, 7.0)
    w = tl.lattice.D3Q19.W_EXACT64.to("cuda:0").reshape(19, 1, 1, 1)
    for i, e in enumerate(edges):
        p = (e * e + 63) // 64 * 64
        v = want.as_strided((19, e, e, e), (p, 19 * p, e, 1), shift + c.offset(i))
        v.copy_((torch.zeros_like(w) if deviation else w).expand_as(v))
    assert torch.equal(buf, want)
