"""run() goes through step() / step2() wherever these are not the class's own (no GPU)."""

from __future__ import annotations

import pytest
import torch

import tensorlbm_amd as tl


def _solver(cls, two):
    s = object.__new__(cls)
    s._two_step, s._report_step = two, 0
    return s


@pytest.mark.parametrize("how", ["class", "instance", "subclass"])
@pytest.mark.parametrize("two", [False, True])
def test_run_calls_a_replaced_step(monkeypatch, how, two):
    calls = []

    def step(self, f, *, force=None):
        calls.append(1)
        return f + 1

    def step2(self, f, *, force=None):
        calls.append(2)
        return f + 2

    cls = tl.FusedSolver3D
    if how == "subclass":
        cls = type("Sub", (cls,), {"step": step, "step2": step2})
    elif how == "class":
        monkeypatch.setattr(cls, "step", step)
        monkeypatch.setattr(cls, "step2", step2)
    s = _solver(cls, two)
    if how == "instance":
        s.step, s.step2 = step.__get__(s), step2.__get__(s)
    f, diags = s.run(torch.zeros(1), 5)
    assert float(f) == 5 and diags == [{}] * 5 and s._report_step == 5
    assert calls == ([2, 2, 1] if two else [1] * 5)
