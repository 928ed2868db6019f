"""The switches that ask for the row walks reach the rule that sends pairs of scales to tiles (no GPU).

The planes are the same bits on either kernel, so only the rule itself can tell; it is called under its
exported C++ name, pms::tile2_range(int h, int w, int scale, int jobs, bool masked, bool recomposition).
"""

import ctypes

import pytest

from pymoresane_amd import _lib

SWITCHES = ("PMS_IUWT_SMALL_LAUNCH", "PMS_IUWT_DEC2", "PMS_IUWT_PAIR")


def _tiles(recomposition, n=1024, jobs=1, masked=False, scale=0):
    rule = _lib.load()._ZN3pms11tile2_rangeEiiiibb
    rule.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool] * 2
    rule.restype = ctypes.c_bool
    return rule(n, n, scale, jobs, masked, recomposition)


@pytest.mark.parametrize("switch,value,decomposition,recomposition", [
    (None, None, True, True), ("PMS_IUWT_SMALL_LAUNCH", "0", False, False),
    ("PMS_IUWT_SMALL_LAUNCH", "8388608", True, True), ("PMS_IUWT_DEC2", "1", False, True),
    ("PMS_IUWT_DEC2", "0", False, True), ("PMS_IUWT_PAIR", "1", True, False), ("PMS_IUWT_PAIR", "0", True, False)])
def test_switches_keep_planes_on_the_walks(monkeypatch, switch, value, decomposition, recomposition):
    for s in SWITCHES:
        monkeypatch.delenv(s, raising=False)
    if switch:
        monkeypatch.setenv(switch, value)
    assert _tiles(False) == decomposition
    assert _tiles(True) == recomposition


@pytest.mark.parametrize("n,jobs,scale,plain,masked", [
    (1024, 4, 0, (True, True), (True, True)), (1024, 4, 2, (True, True), (True, True)),
    (1024, 5, 2, (False, False), (False, False)), (1024, 7, 0, (True, True), (True, True)),
    (1024, 8, 0, (True, True), (False, True)), (1024, 9, 0, (True, True), (False, False)),
    (2048, 3, 0, (True, True), (False, False)), (4096, 1, 0, (False, False), (False, False))])
def test_masked_launches_leave_the_tiles_sooner(monkeypatch, n, jobs, scale, plain, masked):
    for s in SWITCHES:
        monkeypatch.delenv(s, raising=False)
    assert (_tiles(False, n, jobs, False, scale), _tiles(True, n, jobs, False, scale)) == plain
    assert (_tiles(False, n, jobs, True, scale), _tiles(True, n, jobs, True, scale)) == masked
