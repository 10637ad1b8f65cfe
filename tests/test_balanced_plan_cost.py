"""The balanced launch's plan prices what a split costs: a workgroup's fixed
time and the partial results, not only its share of a round."""

from __future__ import annotations

import ctypes

import pytest

from repercep_runtime_amd import _capi


@pytest.mark.parametrize("shape,want", [
    # 224 of 1760 workgroups past six whole rounds: split eight ways they
    # would fill seven eighths of a round, each with its fixed time again; 96
    # past three rounds split two ways, not four or eight
    ((1, 32, 14080, 14080, 128), (55, 1)),
    ((1, 24, 9000, 9000, 128), (32, 2)),
    # a few workgroups past whole rounds, or long key ranges, still split
    ((1, 32, 33000, 33000, 128), (128, 8)),
    ((1, 40, 75600, 75600, 128), (288, 4)),
    ((1, 32, 56320, 56320, 128), (216, 2)),
])
def test_plan(shape: tuple, want: tuple) -> None:
    m, s = ctypes.c_int(), ctypes.c_int()
    assert _capi.lib().rp_fp8_attn_balanced_plan(*shape, 0, 256, ctypes.byref(m),
                                                 ctypes.byref(s)) == 0
    assert (m.value, s.value) == want


@pytest.mark.parametrize("shape,want", [
    # at head dim 256 and 64 the tiles' times, and so what a workgroup's fixed
    # cost and the parts are worth in tiles, are not head dim 128's: us unsplit
    # / split 2, 4, 8 ways
    ((1, 80, 6613, 6613, 256), (24, 2)),      # 2649 / 2573 / 2603 / 2703
    ((1, 40, 12681, 12681, 256), (48, 4)),    # 4503 / 4399 / 4394 / 4415
    ((1, 24, 17343, 17343, 256), (64, 4)),    # 4953 / 4853 / 4839 / 4882
    ((1, 12, 25298, 25298, 256), (96, 8)),    # 5438 / 5172 / 5097 / 5085
    ((1, 8, 12829, 12829, 64), (32, 4)),      # 318 / 333 / 306 / 310
    ((1, 24, 17787, 17787, 64), (64, 8)),     # 1511.5 / 1507.8 / 1465.9 / 1465.6
    ((1, 12, 17713, 17713, 64), (64, 8)),     # 862 / 764 / 763 / 748
    # and these stay unsplit
    ((1, 80, 3538, 3538, 256), (14, 1)),      # 946, four ways 1256
    ((1, 16, 7834, 7834, 64), (31, 1)),       # 1.00 / 1.12 / 1.19 / 1.38
])
def test_plan_per_head_dim(shape: tuple, want: tuple) -> None:
    test_plan(shape, want)
