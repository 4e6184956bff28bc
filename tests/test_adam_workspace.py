"""The optimiser's workspace for single steps exists from the first of them on; epochs have their own (no GPU: the
library's calls are replaced by ones that do nothing)."""

from __future__ import annotations

import types

import pytest
import torch

from tensorlbm_amd import _native as nat
from tensorlbm_amd import closure as cl


class NoLibrary:
    def __getattr__(self, name):
        return lambda *a: 0


def test_workspace_of_single_steps(monkeypatch):
    n = cl.sizes()["nparam"]
    model = types.SimpleNamespace(nparam=n, device=torch.device("cpu"), params=torch.zeros(n), mark_updated=lambda: None)
    opt = cl._Adam(model, 1e-3, max_batch=130)
    monkeypatch.setattr(nat, "lib", lambda: NoLibrary())
    monkeypatch.setattr(nat, "stream_of", lambda t: 0)
    x, t = torch.zeros(300, 7), torch.zeros(300)
    opt.epoch(x, t, torch.arange(300), 128)
    assert opt.t == 3 and opt.partials is None
    opt.step(x[:130], t[:130])
    first = opt.partials
    assert tuple(first.shape) == (3, n + 1)
    opt.step(x[:64], t[:64])
    assert opt.partials is first
    with pytest.raises(ValueError, match="exceeds"):
        opt.step(x[:193], t[:193])
