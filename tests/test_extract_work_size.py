"""The extraction workspace of a plane is large enough for its transpose (no GPU)."""

import pytest

from pymoresane_amd import _lib


@pytest.mark.parametrize("s,h,w", [(1, 1, 1), (2, 601, 1000), (5, 100, 260), (7, 64, 4096), (16, 3, 65)])
def test_extraction_workspace_serves_both_orientations(s, h, w):
    lib = _lib.load()
    assert lib.pms_extract_work_bytes(s, h, w) == lib.pms_extract_work_bytes(s, w, h)
    assert lib.pms_extract_work_bytes(s, h, w) > s * h * w * 4
