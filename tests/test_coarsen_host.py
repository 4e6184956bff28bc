"""Argument checks of the block averages (no GPU): refused before any launch or division."""

from __future__ import annotations

import ctypes

import pytest

from tensorlbm_amd import _native as nat


@pytest.mark.parametrize("dims", [(4, 4, 0), (0, 4, 4), (4, 0, 4), (0, 0, 0), (-4, 4, 4), (4, 4, -4)])
@pytest.mark.parametrize("factor", [1, 2, 600])
def test_empty_grids_are_refused(dims, factor):
    p = ctypes.c_void_p(0x1000)
    assert nat.lib().tlbm_coarsen_moments(19, nat.STORE_F32, p, None, *dims, factor, p, None) == nat.ERR_SHAPE
