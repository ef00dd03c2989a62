"""The layout rule of members that share the GPU, on autotuner reports."""
from snac_amd.ensemble import _ELEM_MS, shared_layout


def _report(*ms):
    return dict(zip(_ELEM_MS, ms))


def test_tet_per_lane_unless_another_is_ten_percent_faster():
    assert shared_layout(_report(0.40, 0.70, 0.71, 0.37)) == 0
    assert shared_layout(_report(0.40, 0.70, 0.71, 0.35)) == 3
    assert shared_layout(_report(0.40, 0.35, 0.34, 0.39)) == 2
    assert shared_layout(_report(0.40, 0.34, 0.35, 0.36)) == 1
    assert shared_layout(_report(0.30, 0.70, 0.71, 0.37)) == 0
