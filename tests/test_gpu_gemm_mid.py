"""The medium-tile GEMM kernel (rp_gemm_mid.h) at its edges: K that ends inside
a 64-byte MFMA depth, ragged M and N, one to many K slices, both ring depths,
split K, both B layouts, bias and row scales -- against the exact product.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from repercep_runtime_amd import _capi as C
from repercep_runtime_amd import ops
from tests._helpers import bf16_bits, bf16_to_f32, codes_np
from tests.test_gemm_plan import plan
from tests.test_gpu_gemm import _assert_one_rounding_apart

pytestmark = pytest.mark.gpu


def _codes(rows: int, cols: int, pad: int, gen: torch.Generator) -> torch.Tensor:
    """(rows, cols) e4m3fn codes as a row-strided view; the `pad` columns after
    each row are NaN codes, which a read past K would turn the result into."""
    wide = torch.full((rows, cols + pad), 0x7F, dtype=torch.uint8)
    wide[:, :cols] = torch.randn(rows, cols, generator=gen).mul(30).to(torch.float8_e4m3fn) \
        .view(torch.uint8)
    return wide


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (1, 16, 16), (64, 128, 80), (65, 144, 144), (128, 272, 208),   # K tails of 16, 16, 16, 16
    (129, 384, 1072), (33, 128, 48), (200, 256, 160),              # 48, 48, 32
    (64, 128, 64), (130, 128, 128), (127, 256, 192), (128, 128, 256),   # whole sub-slices
    (300, 400, 3600),                                              # the P.V product's K
    (16, 512, 4096), (100, 640, 8192), (17, 128, 2064),            # split K
    (70, 144, 2448), (70, 144, 2608), (65, 128, 2624), (128, 256, 2816),   # parts of 4 slices
    (2050, 2064, 208), (2050, 2064, 752),                          # two tiles to a CU
])
def test_edges_vs_exact(gpu: torch.device, M: int, N: int, K: int, bias: bool) -> None:
    g = torch.Generator().manual_seed(M + N + K)
    aw, bw = _codes(M, K, 48, g), _codes(N, K, 16, g)
    assert plan(M, N, K)[0] < 256
    a8, bt8 = aw.to(gpu)[:, :K], bw.to(gpu)[:, :K]
    b = torch.randn(N, generator=g).mul(50).to(torch.bfloat16) if bias else None
    bg = b.to(gpu) if bias else None
    sa, sb = 0.013, 0.0071
    got = ops.fp8_gemm(a8, bt8, sa, sb, b_transposed=True, bias=bg)
    _assert_one_rounding_apart(bf16_to_f32(bf16_bits(got)), None, codes_np(aw[:, :K]),
                               codes_np(bw[:, :K]), sa * sb,
                               b.float().numpy().astype(np.float64) if bias else None)
    # (K, N) row-major: the same bytes in the same order
    kn = torch.full((K, N + 16), 0x7F, dtype=torch.uint8)
    kn[:, :N] = bw[:, :K].t()
    got_kn = ops.fp8_gemm(a8, kn.to(gpu)[:, :N], sa, sb, bias=bg)
    assert torch.equal(got_kn.view(torch.int16), got.view(torch.int16))


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K,tile", [
    (70, 144, 2448, 64), (70, 144, 2608, 64),       # 20 and 21 slices, K tails of 16 and 48
    (65, 128, 2624, 64), (128, 256, 2816, 64),      # whole sub-slices: 41 and 44
    (64, 128, 5120, 64),                            # 40 slices: the ring more than four times
    (500, 5104, 2576, 128), (512, 5104, 2688, 128),   # 160 workgroups, ragged and not
])
def test_four_ahead_ring_vs_exact(gpu: torch.device, M: int, N: int, K: int, tile: int,
                                  bias: bool) -> None:
    """At most a workgroup per CU and 20 or more K slices in one part: the ring
    that loads four slices ahead, through rp_fp8_linear (no workspace, so no
    split), both layouts; NaN codes lie past K and N."""
    assert plan(M, N, K, 1, 0) == (tile, 1, 4)
    g = torch.Generator().manual_seed(M + N + K)
    aw, bw = _codes(M, K, 48, g), _codes(N, K, 16, g)
    kn = torch.full((K, N + 16), 0x7F, dtype=torch.uint8)
    kn[:, :N] = bw[:, :K].t()
    a8, bt8, kn8 = (t.to(gpu) for t in (aw, bw, kn))
    b = torch.randn(N, generator=g).mul(50).to(torch.bfloat16) if bias else None
    bg = b.to(gpu) if bias else None
    outs = []
    for b8, lay in ((bt8, C.RP_B_NK), (kn8, C.RP_B_KN)):
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=gpu)
        C.check(C.lib().rp_fp8_linear(
            a8.data_ptr(), b8.data_ptr(), lay, bg.data_ptr() if bias else None, out.data_ptr(),
            M, N, K, a8.stride(0), b8.stride(0), N, 0.013, 0.0071, None, None, ops._stream(a8)),
            "rp_fp8_linear")
        outs.append(out)
    rows = np.unique(np.linspace(0, M - 1, 40).astype(int))
    _assert_one_rounding_apart(bf16_to_f32(bf16_bits(outs[0]))[rows], None,
                               codes_np(aw[:, :K])[rows], codes_np(bw[:, :K]), 0.013 * 0.0071,
                               b.float().numpy().astype(np.float64) if bias else None)
    assert not bool(torch.isnan(outs[0]).any())
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


def test_split_shapes_split(gpu: torch.device) -> None:
    """The workspace says which products split K: few rows, deep K."""
    L = C.lib()
    base = C.RP_GEMM_BALANCED_WORKSPACE_BYTES
    for M, N, K in ((16, 512, 4096), (100, 640, 8192), (17, 128, 2064)):
        extra = L.rp_fp8_linear_workspace_bytes(M, N, K) - base
        assert extra > 0 and extra % (4 * M * N) == 0 and extra // (4 * M * N) >= 2
    for M, N, K in ((512, 5120, 5120), (75600, 13824, 5120), (64, 128, 256)):
        assert L.rp_fp8_linear_workspace_bytes(M, N, K) == base
    assert L.rp_fp8_linear_workspace_bytes(0, 128, 128) == 0


def test_small_workspace_runs_unsplit(gpu: torch.device) -> None:
    """A product that would split K runs with the counter-sized workspace too,
    unsplit: rp_fp8_linear's bits; the split form's differ from them by its
    order of the sums, and lie as near to the exact product."""
    M, N, K = 32, 512, 4096
    g = torch.Generator(device=gpu).manual_seed(1)
    assert plan(M, N, K)[1] > 1
    a8 = torch.randint(0, 126, (M, K), generator=g, device=gpu, dtype=torch.uint8)
    b8 = torch.randint(0, 126, (N, K), generator=g, device=gpu, dtype=torch.uint8)
    # signs at random: the MFMA truncates, and over operands of one sign that
    # adds up (7.3e-5 of sum |a||b| here, in the large tiles too; 5e-7 with signs)
    a8 |= torch.randint(0, 2, (M, K), generator=g, device=gpu, dtype=torch.uint8) << 7
    outs = [torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=gpu) for _ in range(2)]
    ws = torch.empty(C.RP_GEMM_BALANCED_WORKSPACE_BYTES, dtype=torch.uint8, device=gpu)
    args = (M, N, K, K, K, N, 0.01, 0.02, None, None)
    C.check(C.lib().rp_fp8_linear(a8.data_ptr(), b8.data_ptr(), C.RP_B_NK, None,
                                  outs[0].data_ptr(), *args, ops._stream(a8)), "rp_fp8_linear")
    C.check(C.lib().rp_fp8_linear_balanced(a8.data_ptr(), b8.data_ptr(), C.RP_B_NK, None,
                                           outs[1].data_ptr(), *args, ws.data_ptr(), ws.numel(),
                                           ops._stream(a8)), "rp_fp8_linear_balanced")
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    for c in (outs[0], ops.fp8_gemm(a8, b8, 0.01, 0.02, b_transposed=True)):
        _assert_one_rounding_apart(bf16_to_f32(bf16_bits(c)), None, codes_np(a8.cpu()),
                                   codes_np(b8.cpu()), 0.01 * 0.02)


def test_output_stride_and_untouched_padding(gpu: torch.device) -> None:
    """Row-strided C, 8-byte but not 16-byte aligned rows: the padding stays."""
    M, N, K = 130, 132, 272
    g = torch.Generator().manual_seed(9)
    aw, bw = _codes(M, K, 0, g), _codes(N, K, 0, g)
    a8, bt8 = aw.to(gpu), bw.to(gpu)
    ref = ops.fp8_gemm(a8, bt8, 0.01, 0.01, b_transposed=True)
    wide = torch.full((M, N + 12), 7.0, dtype=torch.bfloat16, device=gpu)
    ops.fp8_gemm(a8, bt8, 0.01, 0.01, b_transposed=True, out=wide[:, 4:4 + N])
    assert torch.equal(wide[:, 4:4 + N], ref)
    assert (wide[:, :4] == 7.0).all() and (wide[:, 4 + N:] == 7.0).all()


@pytest.mark.parametrize("Z,M,N,K", [(2, 200, 128, 400), (3, 129, 64, 3600), (2, 300, 304, 128),
                                     (1, 65, 96, 16), (50, 200, 300, 16), (50, 200, 300, 400)])
def test_row_scaled_batches(gpu: torch.device, Z: int, M: int, N: int, K: int) -> None:
    """Row scales and batch strides: powers of two and small integers, exact."""
    g = torch.Generator().manual_seed(Z + M + N + K)
    a = torch.randint(-2, 3, (Z, M, K), generator=g).float()
    b = torch.randint(-2, 3, (Z, N, K), generator=g).float()
    sa = 2.0 ** torch.randint(-4, 4, (Z, M), generator=g).float()
    sb = 2.0 ** torch.randint(-4, 4, (Z, N), generator=g).float()
    got = ops.gemm_rowwise(a.to(torch.float8_e4m3fn).to(gpu), b.to(torch.float8_e4m3fn).to(gpu),
                           sa.to(gpu), sb.to(gpu)).cpu()
    want = ((a @ b.transpose(1, 2)) * sa[:, :, None] * sb[:, None, :]).to(torch.bfloat16)
    assert torch.equal(got, want)


def test_many_tiles_ragged_edges(gpu: torch.device) -> None:
    """A grid of many rounds (6,825 tiles), ragged in M and N, with a half K
    slice: sampled rows against the exact product."""
    M, N, K = 8200, 13332, 192
    assert plan(M, N, K) == (128, 1, 2)
    g = torch.Generator().manual_seed(3)
    aw, bw = _codes(M, K, 0, g), _codes(N, K, 0, g)
    got = ops.fp8_gemm(aw.to(gpu), bw.to(gpu), 0.01, 0.01, b_transposed=True)
    rows = np.array([0, 1, 255, 256, 4095, 8191, 8192, 8199])
    _assert_one_rounding_apart(bf16_to_f32(bf16_bits(got[torch.from_numpy(rows).to(gpu)])), None,
                               codes_np(aw)[rows], codes_np(bw), 1e-4)
