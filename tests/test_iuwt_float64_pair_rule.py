"""Which scales of a float64 transform run two a launch (no GPU): pms::gen_pair_applies(h, w, scale, jobs, recomposition).

Pairs whose phases have few positions waste most of a 16 x 16 tile: with every pair in one launch, all scales of a
1024^2 or 4096^2 plane took 1.3 to 2.1 times as long as one scale a launch.
"""

import ctypes

import pytest

from pymoresane_amd import _lib


@pytest.mark.parametrize("h,w,scale,jobs,decomposition,recomposition", [
    (64, 64, 4, 1, True, True), (64, 64, 4, 16, False, False), (256, 256, 4, 1, True, True), (256, 256, 6, 1, False, False),
    (512, 512, 4, 1, True, True), (512, 512, 5, 1, True, False), (1024, 1024, 5, 1, True, True),
    (1024, 1024, 6, 1, True, False), (1024, 1024, 8, 1, False, False), (4096, 4096, 7, 1, True, True),
    (4096, 4096, 10, 1, False, False), (64, 4096, 3, 1, False, False), (512, 512, 8, 1, False, False)])
def test_pairs_need_phases_that_fill_a_tile(h, w, scale, jobs, decomposition, recomposition):
    applies = _lib.load()._ZN3pms16gen_pair_appliesEiiiib
    applies.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool]
    applies.restype = ctypes.c_bool
    assert applies(h, w, scale, jobs, False) == decomposition
    assert applies(h, w, scale, jobs, True) == recomposition
