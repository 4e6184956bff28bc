"""Host time of two-step launches of small lattices stepped in turn (no GPU: the launch itself is an error here)."""

from __future__ import annotations

import ctypes
import time

import pytest
import torch

from tensorlbm_amd import _native as nat


@pytest.mark.skipif(torch.cuda.is_available(), reason="times the call up to a launch that fails")
@pytest.mark.parametrize("n", [2, 8, 16])
def test_lattices_in_turn_cost_what_one_costs(n):
    """The launch shape of each is found once, not again at every change of lattice (5 - 20 us each time)."""
    lib, coll = nat.lib(), nat.make_collision(nat.COLL_BGK, 0.7)
    a, b = ctypes.c_void_p(0x100000), ctypes.c_void_p(0x900000)

    def per_call(shapes):
        best = float("inf")
        for _ in range(200):
            t = time.perf_counter()
            for s in shapes:
                assert lib.tlbm_step2(19, nat.STORE_F32, a, None, b, None, *s, coll, None, None, None, None) \
                    == nat.ERR_HIP
            best = min(best, time.perf_counter() - t)
        return best / len(shapes)

    one = per_call([(58, 57, 55)] * 16)
    assert per_call([(58 + i, 57, 55 - i) for i in range(n)] * (16 // n)) <= 1.5 * one + 2e-6
