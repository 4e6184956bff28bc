"""Outputs of the eager operators are plain contiguous tensors whatever the input is (no GPU: the library's calls
are replaced by ones that do nothing)."""

from __future__ import annotations

import pytest
import torch

import tensorlbm_amd as tl
from tensorlbm_amd import _native as nat


class NoLibrary:
    def __getattr__(self, name):
        return lambda *a: 0


class Tagged(torch.Tensor):
    pass


@pytest.fixture(autouse=True)
def no_gpu(monkeypatch):
    monkeypatch.setattr(nat, "lib", lambda: NoLibrary())
    monkeypatch.setattr(nat, "require_gpu", lambda t, what: None)
    monkeypatch.setattr(nat, "stream_of", lambda t: 0)


OPS = [(tl.macroscopic, 9), (tl.stream, 9), (tl.macroscopic3d, 19), (tl.stream3d, 19), (tl.macroscopic27, 27),
       (tl.stream27, 27)]


def _outputs(op, f):
    out = op(f)
    return out if isinstance(out, (tuple, list)) else [out]


@pytest.mark.parametrize("op,q", OPS)
def test_subclass_in_plain_tensor_out(op, q):
    shape = (q, 4, 5) if q == 9 else (q, 3, 4, 5)
    for cls in (Tagged, torch.nn.Parameter):
        f = torch.zeros(shape)
        f = f.as_subclass(Tagged) if cls is Tagged else cls(f)
        for o in _outputs(op, f):
            assert type(o) is torch.Tensor and not o.requires_grad


@pytest.mark.parametrize("op,q", OPS)
def test_odd_strides_of_single_cell_axes(op, q):
    """An axis of one cell may have any stride in a contiguous tensor; the outputs have the standard ones."""
    shape = (q, 1, 5) if q == 9 else (q, 3, 1, 5)
    buf = torch.zeros(q * 15)
    stride = (5, 777, 1) if q == 9 else (15, 5, 777, 1)
    f = buf.as_strided(shape, stride)
    assert f.is_contiguous()
    for o in _outputs(op, f):
        assert o.stride() == torch.empty(o.shape).stride()
