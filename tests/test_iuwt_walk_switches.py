"""The switches that ask for the row walks reach the rule that sends pairs of scales to tiles (no GPU).

The planes are the same bits on either kernel, so only the rule itself can tell; it is called under its
exported C++ name, pms::tile2_range(int h, int w, int scale, int jobs, bool recomposition).
"""

import pytest

from pymoresane_amd import _lib

SWITCHES = ("PMS_IUWT_SMALL_LAUNCH", "PMS_IUWT_DEC2", "PMS_IUWT_PAIR")


def _tiles(recomposition):
    import ctypes
    rule = _lib.load()._ZN3pms11tile2_rangeEiiiib
    rule.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool]
    rule.restype = ctypes.c_bool
    return rule(1024, 1024, 0, 1, recomposition)


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
