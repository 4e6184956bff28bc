"""Tensors that torch must see written: the one-launch companions of the obstacle step write through addresses only
where torch's in-place operators would do nothing else, and say so to autograd.

On the CPU the library is replaced by one whose calls only count; on the GPU it is the real one."""

from __future__ import annotations

import pytest
import torch
import torch.autograd.forward_ad as fw
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

import tensorlbm_amd as tl
from tensorlbm_amd import _native as nat
from tensorlbm_amd import fused

SHAPE = (19, 6, 4, 5)
GPU = pytest.param("cuda:0", marks=pytest.mark.gpu)


class CountingLibrary:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *a: self.calls.append(name) or 0


@pytest.fixture(params=["cpu", GPU])
def where(request, monkeypatch):
    """(device, list of library calls or None)"""
    if request.param != "cpu":
        return request.param, None
    lib = CountingLibrary()
    monkeypatch.setattr(nat, "lib", lambda: lib)
    monkeypatch.setattr(nat, "require_gpu", lambda t, what: None)
    monkeypatch.setattr(nat, "stream_of", lambda t: 0)
    monkeypatch.setattr(nat, "on_current_device", lambda t: True, raising=False)
    return "cpu", lib.calls


def _state(device, seed=0, shape=SHAPE):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(device)


def _planes(f, feq):
    face = feq[:, None, None]
    f[:, :, :, 0] = face
    f[:, :, :, -1] = f[:, :, :, -2]
    f[:, :, 0, :] = face
    f[:, :, -1, :] = face
    f[:, 0] = face
    f[:, -1] = face
    return f


@pytest.mark.parametrize("dual", ["f", "feq"])
def test_faces_carry_tangents(where, dual):
    device, calls = where
    f, feq = _state(device), _state(device, 1)[:, 0, 0, 0].contiguous()
    with fw.dual_level():
        pair = {"f": f, "feq": feq}
        tangent = _state(device, 2) if dual == "f" else _state(device, 2)[:, 1, 1, 1].contiguous()
        pair[dual] = fw.make_dual(pair[dual].clone(), tangent.clone())
        tl.apply_far_field_bc_6face(pair["f"], 0.05, feq_vec=pair["feq"])
        got = fw.unpack_dual(pair["f"])
        want = _planes(tangent.clone(), torch.zeros_like(feq)) if dual == "f" else _planes(torch.zeros_like(f), tangent)
        assert torch.equal(got.tangent, want)
        assert torch.equal(got.primal, _planes(f.clone(), feq))
    assert not calls


def test_faces_under_vmap(where):
    device, calls = where
    f, feq = _state(device, shape=(3,) + SHAPE), _state(device, 1)[:, 0, 0, 0].contiguous()
    want = torch.stack([_planes(x.clone(), feq) for x in f])

    def faces(x):
        tl.apply_far_field_bc_6face(x, 0.05, feq_vec=feq)
        return x

    assert torch.equal(torch.vmap(faces)(f), want)
    assert not calls


def test_faces_seen_by_modes_and_tracers(where):
    device, calls = where
    feq = _state(device, 1)[:, 0, 0, 0].contiguous()

    class Log(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Log.ops += func is torch.ops.aten.copy_.default
            return func(*args, **(kwargs or {}))

    f = _state(device)
    with Log():
        tl.apply_far_field_bc_6face(f, 0.05, feq_vec=feq)
    assert Log.ops == 6

    def faces(x):
        x = x.clone()
        tl.apply_far_field_bc_6face(x, 0.05, feq_vec=feq)
        return x

    g = make_fx(faces)(_state(device))
    for seed in (3, 4):
        x = _state(device, seed)
        assert torch.equal(g(x), _planes(x.clone(), feq))
    assert not calls


def test_inference_tensors_stay_refused(where):
    device, calls = where
    with torch.inference_mode():
        f = _state(device)
    with pytest.raises(RuntimeError, match="inference tensor"):
        tl.apply_far_field_bc_6face(f, 0.05, feq_vec=f[:, 0, 0, 0].clone())
    with pytest.raises(RuntimeError, match="inference tensor"):
        _force(f.clone(), [f[i, 0, 0, :1] for i in range(3)], None)
    assert not calls


def _force(f, bufs, monkeypatch):
    """A force sample of (1, 2, 3) added to the buffers."""
    real = fused._launch_step
    fused._launch_step = lambda f, out, coll, solid=None, force=None, what="": force.copy_(
        torch.tensor([1.0, 2.0, 3.0], dtype=torch.float64))
    try:
        tl.fused_obstacle_step(f, 0.02, torch.zeros(f.shape[1:], dtype=torch.int8, device=f.device), 0.0, 1.0,
                               fx_buf=bufs[0], fy_buf=bufs[1], fz_buf=bufs[2])
    finally:
        fused._launch_step = real


def test_force_buffers_carry_tangents(where):
    device, calls = where
    with fw.dual_level():
        t = [torch.full((1,), 0.5 + i, device=device) for i in range(3)]
        bufs = [fw.make_dual(torch.full((1,), float(i), device=device), t[i]) for i in range(3)]
        _force(_state(device), bufs, None)
        for i, b in enumerate(bufs):
            d = fw.unpack_dual(b)
            assert float(d.primal) == 2.0 * i + 1.0 and float(d.tangent) == 0.5 + i
    assert not calls


def test_saved_tensors_notice_the_launch(where):
    device, calls = where
    f, feq = _state(device), _state(device, 1)[:, 0, 0, 0].contiguous()
    w = torch.ones((), device=device, requires_grad=True)
    for given in ({"feq_vec": feq}, {}):  # both forms of the launch
        loss = (w * f).sum()
        tl.apply_far_field_bc_6face(f[:, :, :, :], 0.05, **given)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            loss.backward()
    bufs = [torch.ones(1, device=device) for _ in range(3)]
    loss = sum((w * b).sum() for b in bufs)
    versions = [b._version for b in bufs]
    _force(f, bufs, None)
    assert [b._version for b in bufs] == [v + 1 for v in versions]
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()
    assert calls is None or calls == ["tlbm_far_field_faces", "tlbm_far_field_faces", "tlbm_force_add"]


def test_launches_in_inference_mode(where):
    device, calls = where
    with torch.inference_mode():
        f = _state(device)
        tl.apply_far_field_bc_6face(f, 0.05, feq_vec=f[:, 0, 0, 0].clone())
        _force(f, [f[i, 0, 0, :1].clone() for i in range(3)], None)
    assert calls is None or calls == ["tlbm_far_field_faces", "tlbm_force_add"]


@pytest.mark.parametrize("shape", [(19, 2, 2, 2**29), (65536, 2, 2, 3)])
def test_faces_beyond_the_launch_limits(monkeypatch, shape):
    """2^31 cells (82 GB in half precision) or 65536 populations: more than the launch takes, plane by plane then."""
    lib = CountingLibrary()
    monkeypatch.setattr(nat, "lib", lambda: lib)
    monkeypatch.setattr(nat, "require_gpu", lambda t, what: None)
    monkeypatch.setattr(nat, "stream_of", lambda t: 0)
    monkeypatch.setattr(nat, "on_current_device", lambda t: True)
    f = torch.empty(shape, dtype=torch.float16, device="meta")
    tl.apply_far_field_bc_6face(f, 0.05, feq_vec=torch.empty(19, device="meta"))
    assert not lib.calls
