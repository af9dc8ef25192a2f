"""The work splits the launchers choose, by the library's plan functions (no GPU)."""
import ctypes

import pytest

from fv3core_amd import _lib


def rows_of(march, rows, planes, fp32, *most):
    fn = getattr(_lib.lib(), f"fv3_plan_{march}_rows")
    return fn(rows, ctypes.c_int64(planes), int(fp32), *most)


# Launches of six tiles and 79 levels where a march's own cost and the FP64 del-n
# march's lead to different segments: (march, cells a side, FP32, rows a segment).
@pytest.mark.parametrize("march,n,fp32,seg", [
    ("delnflux", 48, True, 9), ("delnflux", 48, False, 10), ("delnflux", 128, True, 26),
    ("delnflux", 128, False, 65), ("c_sw", 12, False, 5), ("c_sw", 12, True, 5),
    ("c_sw", 24, False, 8), ("c_sw", 96, False, 35), ("d2a2c", 12, False, 5),
    ("d2a2c", 24, False, 5)])
def test_each_march_splits_by_its_own_cost(march, n, fp32, seg):
    beside, width = {"delnflux": (1, 58), "c_sw": (7, 62), "d2a2c": (6, 60)}[march]
    rows = n + beside
    planes = -(-rows // width) * 6 * 79
    most = (0,) if march == "delnflux" else ()
    assert rows_of(march, rows, planes, fp32, *most) == seg


@pytest.mark.parametrize("march", ["delnflux", "c_sw", "d2a2c"])
@pytest.mark.parametrize("fp32", [False, True])
def test_segments_stay_within_the_rows(march, fp32):
    most = (0,) if march == "delnflux" else ()
    for rows in (1, 2, 3, 4, 7, 33, 49, 97, 200, 1001):
        for planes in (1, 6, 474, 3072, 7584, 300000):
            seg = rows_of(march, rows, planes, fp32, *most)
            assert 1 <= seg <= rows
            if planes > 3 * 1024:  # more than three waves a SIMD however they are cut
                assert seg <= 33


@pytest.mark.parametrize("n", [12, 48, 96, 128, 384])
def test_a2b_segments_keep_the_cap_on_every_launch(n):
    rows = n - 1
    planes = -(-rows // 58) * 6 * 79
    seg = rows_of_a2b(rows, planes, 0)
    assert 1 <= seg <= 33
    assert 1 <= rows_of_a2b(rows, planes, 17) <= 17


def rows_of_a2b(rows, planes, most):
    return _lib.lib().fv3_plan_a2b_rows(rows, ctypes.c_int64(planes), most)
