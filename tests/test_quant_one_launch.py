"""Which Q/K/V quantizer calls run in one launch: not those whose groups leave
most of a workgroup's threads idle and are many, and inside a captured graph
not those that one CU per group makes slower than two launches.  Either form
writes the same scales and codes."""

from __future__ import annotations

import ctypes

import pytest
import torch

from repercep_runtime_amd import _capi, ops


@pytest.mark.parametrize("groups,elems,tiles,eager,captured", [
    (8, 65536, 8, 1, 0),       # a whole group per CU, 24 of 256 busy
    (31, 65536, 8, 1, 0), (32, 65536, 8, 1, 1), (1280, 65536, 8, 1, 1),
    (8, 32768, 4, 1, 1), (8, 32769, 4, 1, 0), (8, 32768, 5, 1, 0), (640, 32768, 4, 1, 1),
    (2560, 16384, 2, 1, 1), (2560, 16383, 2, 0, 0),
    (170, 8192, 1, 1, 1), (171, 8192, 1, 0, 0), (8, 8191, 1, 1, 0),
    (170, 64, 1, 1, 0), (171, 64, 1, 0, 0), (2560, 1024, 1, 0, 0),
])
def test_rule(groups: int, elems: int, tiles: int, eager: int, captured: int) -> None:
    L = _capi.lib()
    assert L.rp_selftest_quant_one_launch(groups, elems, tiles, 0) == eager
    assert L.rp_selftest_quant_one_launch(groups, elems, tiles, 1) == captured


def _kernels(graph: torch.cuda.CUDAGraph) -> int:
    """Kernel nodes of a captured graph (the HIP runtime is a dependency of the library)."""
    L = _capi.lib()
    n = ctypes.c_size_t()
    raw = ctypes.c_void_p(graph.raw_cuda_graph())
    assert L.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert L.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    kind, count = ctypes.c_int(), 0
    for node in nodes:
        assert L.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        count += kind.value == 0      # hipGraphNodeTypeKernel
    return count


@pytest.mark.gpu
@pytest.mark.parametrize("H,S,D,launches", [
    (8, 1024, 64, 2), (40, 512, 128, 1), (8, 256, 128, 1), (4, 64, 64, 2), (300, 16, 128, 2),
])
def test_captured_launches_and_bits(gpu: torch.device, H: int, S: int, D: int,
                                    launches: int) -> None:
    g = torch.Generator(device=gpu).manual_seed(H + S)
    q, k, v = (torch.randn((1, H, S, D), generator=g, device=gpu).to(torch.bfloat16)
               for _ in range(3))
    want = [t.clone() for t in ops.scale_quantize_qkv(q, k, v)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        got = ops.scale_quantize_qkv(q, k, v)
    assert _kernels(graph) == launches
    graph.instantiate()
    for _ in range(3):
        for t in got:
            t.view(torch.uint8).zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
