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
