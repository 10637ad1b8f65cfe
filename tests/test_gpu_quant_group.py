"""The one-launch Q/K/V quantizer for groups that fit a workgroup's registers:
scales, codes and V^T padding equal the single-tensor calls' (amax, finalize
and apply launches) bit for bit, up to and past the sizes it is chosen for."""

from __future__ import annotations

import pytest
import torch

from repercep_runtime_amd import ops

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Sq, Skv, D, dtype, granularity, (B, S, H, D) buffers
    (1, 8, 1024, 1024, 64, torch.bfloat16, "bh", False),     # 65536 elements: the largest group
    (1, 3, 512, 512, 128, torch.float16, "bh", True),        # as many, strided
    (1, 3, 513, 500, 128, torch.bfloat16, "bh", False),      # Q one row past it
    (1, 3, 500, 513, 128, torch.bfloat16, "bh", True),       # K and V past it
    (2, 5, 77, 301, 64, torch.bfloat16, "bh", True),
    (2, 2, 1, 1, 32, torch.bfloat16, "bh", False),           # one row, half-wide V^T tile
    (1, 4, 1024, 1023, 32, torch.float16, "bh", True),       # 8 V^T tiles of 32 columns
    (1, 4, 300, 1025, 32, torch.bfloat16, "bh", False),      # 9 tiles
    (1, 2, 256, 255, 256, torch.bfloat16, "bh", True),       # four column tiles
    (2, 3, 65, 33, 128, torch.bfloat16, "tensor", True),     # one group over six heads, 12 tiles
    (2, 2, 65, 129, 64, torch.bfloat16, "tensor", True),     # one group over four heads
    (1, 1, 500, 900, 64, torch.float16, "tensor", False),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + f"-{c[6]}")
def test_equals_single_tensor_calls(gpu: torch.device, case: tuple) -> None:
    B, H, Sq, Skv, D, dtype, gran, permuted = case
    g = torch.Generator(device=gpu).manual_seed(sum(case[:5]))

    def make(S: int, scale: float) -> torch.Tensor:
        if permuted:
            x = torch.randn((B, S, H, D), generator=g, device=gpu).mul(scale).to(dtype)
            return x.permute(0, 2, 1, 3)
        return torch.randn((B, H, S, D), generator=g, device=gpu).mul(scale).to(dtype)

    q, k, v = make(Sq, 3.0), make(Skv, 0.2), make(Skv, 1.0)
    if gran == "bh" and H > 1:
        q[0, 0] = 0                                   # a zero head
        k[0, 1, 0, 0] = float("inf")                  # an infinite element
        v[0, 1, Skv - 1, D - 1] = float("nan")        # a NaN head: its padding stays 0
    got = ops.scale_quantize_qkv(q, k, v, gran)
    for x, s, c, lay in ((q, got[0], got[1], "bhsd"), (k, got[2], got[3], "bhsd"),
                         (v, got[4], got[5], "bhds")):
        dq, codes = ops.scale_quantize(x, gran, lay)
        assert torch.equal(s.view(torch.int32)[~s.isnan()], dq.view(torch.int32)[~dq.isnan()])
        assert torch.equal(s.isnan(), dq.isnan())
        a, b = c.view(torch.uint8), codes.view(torch.uint8)
        nan = (b & 0x7F) == 0x7F                      # a NaN code's sign is not specified
        assert torch.equal(a[~nan], b[~nan]) and bool(((a[nan] & 0x7F) == 0x7F).all())
        if lay == "bhds":
            assert bool((a[..., Skv:] == 0).all())


@pytest.mark.parametrize("rows", [1, 511, 512, 513])
@pytest.mark.parametrize("gran", ["tensor", "bh"])
def test_single_tensor_scale_and_codes_around_the_fold(gpu: torch.device, rows: int,
                                                       gran: str) -> None:
    """One tensor with up to 256 partial maxima per group folds them in the
    apply launch (512 rows of 8192), one more runs the finalize launch: both
    equal the scale and the codes of separate calls."""
    g = torch.Generator(device=gpu).manual_seed(rows)
    for permuted in (False, True):
        x = torch.randn((1, rows, 2, 8192) if permuted else (1, 2, rows, 8192), generator=g,
                        device=gpu).to(torch.bfloat16)
        x = x.reshape(1, rows, 2 * 8, 1024).permute(0, 2, 1, 3) if permuted else x
        dq, codes = ops.scale_quantize(x, gran)
        ref = ops.per_bh_scale(x, gran)
        assert torch.equal(dq, ref)
        assert torch.equal(codes.view(torch.uint8), ops.quantize(x, ref, gran).view(torch.uint8))
