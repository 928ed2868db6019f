"""Which pairs of scales run on 32 x 32 tiles (no GPU): pms::tile2_fits(h, w, scale, jobs, recomposition).

A recomposition whose phases have at most 16 rows keeps the 16 x 16 tiles (7 to 11% faster there); the same planes'
decompositions, the turned planes and those with more rows take the larger ones.
"""

import ctypes

import pytest

from pymoresane_amd import _lib


@pytest.mark.parametrize("h,w,scale,decomposition,recomposition", [
    (64, 2048, 2, True, False), (64, 4096, 3, True, False), (256, 2048, 4, True, False), (68, 2048, 2, True, True),
    (2048, 64, 2, True, True), (601, 1000, 2, True, True), (1024, 1024, 0, True, True), (256, 256, 0, False, False)])
def test_recompositions_of_flat_phases_keep_the_small_tiles(h, w, scale, decomposition, recomposition):
    fits = _lib.load()._ZN3pms10tile2_fitsEiiiib
    fits.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool]
    fits.restype = ctypes.c_bool
    assert fits(h, w, scale, 1, False) == decomposition
    assert fits(h, w, scale, 1, True) == recomposition
