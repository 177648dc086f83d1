"""Slots of the output levels: as ``i in levels`` finds them, level by level
(src/bldfm/solver.py:189-190), for every form that levels come in."""

import numpy as np
import pytest

from bldfm_amd.solver import _level_maps

FORMS = [
    [1, 2], [0], [3, 3, 1], [-1, 2], [1.0, 2.5], [float("nan"), 2.0], (1, 2), range(3), [1 + 0j, 2], ["1"], [2**70, 3],
    np.array([1, 2], np.uint8), np.array([1, 300], np.int16), np.array([1.0, 5.0], np.float32), np.array([2, 7], np.uint64),
    np.array([True, False]), np.array([1, 2], object), np.array([2.0**53, 3.0]), np.array([np.inf, 1.0]),
    np.array([3, 2048], np.float16), np.ma.array([1, 2], mask=[0, 1]), np.ma.array([1.0, 2.0], mask=[1, 0]),
]


@pytest.mark.parametrize("levels", FORMS, ids=[repr(f)[:40].replace("\n", " ") for f in FORMS])
@pytest.mark.parametrize("nz", [9, 400, 4000])
def test_slots_are_those_of_the_membership_test(levels, nz):
    want = np.full(nz, -1)
    hit = [i for i in range(nz) if i in levels]
    want[hit] = np.arange(len(hit))
    slot, idx = _level_maps(levels, nz)
    assert slot.dtype == np.int32 and np.array_equal(slot, want)
    assert len(idx) == len(levels)
