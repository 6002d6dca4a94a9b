"""The wrappers' scratch under graph capture: a graph keeps what its calls wrote their partial sums to, whatever runs later."""
import pytest
import torch

import gemm_amd as g
import neoGEMM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mod", [g, neoGEMM])
def test_a_graph_keeps_its_scratch(mod):
    gen = torch.Generator(device="cuda").manual_seed(9)

    def ints(*shape):
        return torch.randint(-2, 3, shape, generator=gen, device="cuda").to(torch.bfloat16)

    M, N, K = 264, 392, 8200   # K is split
    need = g.workspace_bytes(M, N, K)
    A, B, large = ints(M, K), ints(K, N), (ints(1024, 16384), ints(16384, 1024))
    assert 0 < need < g.workspace_bytes(1024, 1024, 16384)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        mod.gemm(A, B)   # the kernels are set up, and the stream has a buffer of this size
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        C = mod.gemm(A, B)
    with torch.cuda.stream(stream):
        mod.gemm(*large)   # outgrows that buffer: its block is free for other tensors of this stream
        others = [torch.full((need,), 7, dtype=torch.uint8, device="cuda") for _ in range(4)]
    torch.cuda.synchronize()
    for _ in range(3):
        A.copy_(ints(M, K))
        C.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, mod.gemm(A, B)) and torch.equal(C, (A.float() @ B.float()).to(torch.bfloat16))
        assert all(bool((t == 7).all()) for t in others)
