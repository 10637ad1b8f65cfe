"""Which tiles a product runs on: the medium ones wherever they all run at once,
past that only where they were measured no slower than the large ones."""

from __future__ import annotations

import ctypes

import pytest

from repercep_runtime_amd import _capi


def plan(M: int, N: int, K: int, batch: int = 1, may_split: int = 1) -> tuple[int, int, int]:
    """(tile rows, K parts, slices ahead)"""
    v = [ctypes.c_int() for _ in range(3)]
    assert _capi.lib().rp_fp8_gemm_plan(M, N, K, batch, may_split, *map(ctypes.byref, v)) == 0
    return tuple(x.value for x in v)


@pytest.mark.parametrize("M,N,K,tile", [
    # one round of large tiles: the medium ones took 1.03-1.54 times as long
    (2048, 5120, 13824, 256), (2048, 5120, 5120, 256), (1024, 11008, 4096, 256),
    (700, 13824, 5120, 256), (850, 13824, 5120, 256), (6000, 1536, 8960, 256),
    # several rounds, the last well filled, or weights past the caches: 1.1-1.5 times
    (6000, 5120, 5120, 256), (7000, 5120, 13824, 256), (4096, 5120, 13824, 256),
    (75600, 13824, 5120, 256), (75600, 5120, 5120, 256),
    # a nearly empty last round, or a half empty one: 0.68-0.95
    (8192, 3072, 3072, 128), (6000, 4096, 4096, 128), (1300, 11008, 4096, 128), (3600, 5120, 5120, 128), (6000, 3072, 3072, 128),
    # two medium tiles to a CU, all at once
    (512, 5120, 5120, 128), (2048, 4096, 4096, 128), (1500, 5120, 13824, 128),
    # short K, and K off the large tiles' 64
    (20000, 3072, 512, 128), (75600, 13824, 208, 128),
])
def test_projections(M: int, N: int, K: int, tile: int) -> None:
    assert plan(M, N, K)[0] == tile


@pytest.mark.parametrize("batch,M,N,K,tile", [
    (40, 3600, 3600, 128, 128),      # one latent frame's scores, 0.80
    (40, 3600, 128, 3600, 128),      # and their product with V: K off 64
    (40, 4096, 128, 4096, 128),      # half the columns of a large tile
    (40, 4096, 4096, 1024, 256), (40, 4096, 4096, 2048, 256),   # 1.12, 1.31
    (40, 2500, 2500, 512, 256),      # C rows off 16 bytes, 500 MB of them: 1.14
    (40, 2500, 2504, 512, 128),      # on 16 bytes
    (8, 2500, 2500, 512, 128),       # off, 100 MB: 0.65
])
def test_batches(batch: int, M: int, N: int, K: int, tile: int) -> None:
    assert plan(M, N, K, batch, 0)[0] == tile


def test_ring_depth_and_split() -> None:
    assert plan(512, 5120, 5120) == (128, 1, 4)        # a CU each, 40 slices
    assert plan(2048, 4096, 4096)[2] == 2              # two to a CU
    assert plan(300, 400, 512)[2] == 2                 # few slices
    assert plan(16, 512, 4096)[1] > 1 and plan(16, 512, 4096, may_split=0)[1] == 1


def test_bad_arguments() -> None:
    v = ctypes.c_int()
    L, p = _capi.lib(), ctypes.byref(v)
    for args in ((0, 1, 1, 1, 0), (1, 0, 1, 1, 0), (1, 1, 0, 1, 0), (1, 1, 1, 0, 0)):
        assert L.rp_fp8_gemm_plan(*args, p, p, p) == 1
    assert L.rp_fp8_gemm_plan(1, 1, 1, 1, 0, None, p, p) == 1
