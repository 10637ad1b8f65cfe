"""The longest-first order of causal launches: every (head, query block) runs
exactly once, whatever the head count, the query blocks per head, and the head
dim's halves, on grids just above one round of workgroups and above one chunk
of 32 heads."""

from __future__ import annotations

import pytest
import torch

from repercep_runtime_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Skv,D", [
    (1, 43, 1500, 1500, 64),     # 258 workgroups of 6 blocks, two chunks (32 + 11 heads)
    (2, 19, 1800, 1024, 128),    # 38 heads, keys shorter than queries
    (1, 5, 6700, 6700, 256),     # halves: 270 workgroups, 135 blocks (odd over the XCDs)
    (1, 16, 2304, 2304, 256),    # halves, blocks divide over the XCDs
    (1, 33, 2100, 4000, 32),     # one head in the second chunk
])
def test_causal_rows_equal_their_own_launch(gpu: torch.device, B: int, H: int, Sq: int, Skv: int,
                                            D: int) -> None:
    """Against launches of one head each (one round: the plain order), bit for
    bit: a block's rows do not depend on where it runs."""
    g = torch.Generator(device=gpu).manual_seed(H + Sq)
    q = torch.randn((B, H, Sq, D), generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn((B, H, Skv, D), generator=g, device=gpu).to(torch.bfloat16)
            for _ in range(2))
    out = torch.full_like(q, float("nan"))
    ops.fp8_flash_attention(q, k, v, causal=True, kv_splits=1, out=out)
    for b in range(B):
        for h in range(H):
            one = ops.fp8_flash_attention(q[b:b + 1, h:h + 1], k[b:b + 1, h:h + 1],
                                          v[b:b + 1, h:h + 1], causal=True, kv_splits=1)
            assert torch.equal(one[0, 0].view(torch.int16), out[b, h].view(torch.int16)), (b, h)
