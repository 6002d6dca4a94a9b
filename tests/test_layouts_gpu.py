"""Operands that are transposed views, read in place: both operands with their long side contiguous (A [K,M], B [K,N]) and
A [K,M] beside B [N,K].  Small integers, so that every order of summation gives the same bits."""
import pytest
import torch

import gemm_amd as g
import neoGEMM
from gemm_amd import _abi

pytestmark = pytest.mark.gpu


def small_ints(gen, *shape, top=2):
    return torch.randint(-top, top + 1, shape, generator=gen, device="cuda").to(torch.bfloat16)


def general(A, B, C, M, N, K, lda, ldb, ldc, a_layout, b_layout, c_layout, alpha=1.0, beta=0.0):
    g.gemm_into(A, B, C, M, N, K, lda, ldb, ldc, b_layout, c_layout, alpha=alpha, beta=beta, a_layout=a_layout)


# K: less than a slab, a partial slab, every length of the main loop's prologue, steady state (eight slabs a trip) and tail,
# K that is no multiple of 8 (whole k-rows end anywhere); M, N: edges of the 128 and 256 tiles; deep K with few tiles: split
@pytest.mark.parametrize("M,N,K", [(136, 8, 7), (264, 392, 33), (264, 392, 64), (520, 264, 100), (136, 520, 129), (264, 136, 256), (264, 392, 449),
                                   (392, 264, 640), (264, 392, 1000), (264, 392, 1031), (5128, 5128, 200), (2568, 264, 520), (136, 2056, 6000)])
@pytest.mark.parametrize("b_layout", [g.B_KN, g.B_NK])
@pytest.mark.parametrize("c_layout", [g.C_ROW, g.C_COL])
def test_transposed_a(M, N, K, b_layout, c_layout):
    if b_layout == g.B_NK:
        K = (K + 7) // 8 * 8
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = small_ints(gen, K, M + 8), small_ints(gen, *((K, N + 16) if b_layout == g.B_KN else (N, K)))
    At, Bkn = A[:, :M].t(), (B[:, :N] if b_layout == g.B_KN else B.t())
    want = (At.float() @ Bkn.float())
    C = torch.full((M, N) if c_layout == g.C_ROW else (N, M), float("nan"), dtype=torch.bfloat16, device="cuda")
    general(A, B, C, M, N, K, M + 8, B.stride(0), C.stride(0), g.A_KM, b_layout, c_layout)
    got = C if c_layout == g.C_ROW else C.t()
    assert torch.equal(got, want.to(torch.bfloat16))
    general(A, B, C, M, N, K, M + 8, B.stride(0), C.stride(0), g.A_KM, b_layout, c_layout, alpha=0.5, beta=-1.0)
    assert torch.equal(got, (0.5 * want - want.to(torch.bfloat16).float()).to(torch.bfloat16))


@pytest.mark.parametrize("split", [2, 3, 8])
def test_transposed_a_with_k_split(split):
    """Splits of K over the transposed pair: the plan's own choice on shapes with few tiles, against the unsplit sum."""
    M, N, K = 256, 264, 1024 * split + 72
    gen = torch.Generator(device="cuda").manual_seed(split)
    A, B = small_ints(gen, K, M), small_ints(gen, K, N)
    assert _abi.load().neogemm_bf16_general_workspace_bytes(M, N, K, g.A_KM, g.B_KN, g.C_ROW, 1) > 0
    assert torch.equal(neoGEMM.gemm(A.t(), B), (A.t().float() @ B.float()).to(torch.bfloat16))


@pytest.mark.parametrize("mod", [g, neoGEMM])
def test_wrappers_on_transposed_views(mod):
    """A.t() of what the kernels take in place, and of what they do not (few rows, odd sizes, offset storage): same results."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    for (M, N, K) in ((256, 264, 200), (136, 128, 65), (128, 64, 64), (133, 64, 64), (256, 63, 64), (300, 264, 7)):
        A, B = small_ints(gen, K, M), small_ints(gen, K, N)
        want = (A.t().float() @ B.float())
        assert torch.equal(mod.gemm(A.t(), B), want.to(torch.bfloat16))
        W = small_ints(gen, N, K)
        assert torch.equal(mod.gemm(A.t(), W.t()), (A.t().float() @ W.t().float()).to(torch.bfloat16))
        C = small_ints(gen, M, N)
        sums = (want + C.float()).to(torch.bfloat16)
        mod.gemm_scaled(A.t(), B, C, 1.0, 1.0)
        assert torch.equal(C, sums)
    flat = small_ints(gen, 200 * 256 + 1)
    A, B = flat[1:].view(200, 256), small_ints(gen, 200, 256)
    assert torch.equal(mod.gemm(A.t(), B), (A.t().float() @ B.float()).to(torch.bfloat16))


# several rounds of tiles, the kernels for operands at any address (odd n), copies of them on the 16-byte grid
@pytest.mark.parametrize("n", [264, 515, 2501, 6144])
@pytest.mark.parametrize("mod", [g, neoGEMM])
def test_output_in_the_memory_of_a_transposed_a(mod, n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    C, X = small_ints(gen, n, n), small_ints(gen, n, n)
    want = (C.t().float() @ X.float() + C.float()).to(torch.bfloat16)
    mod.gemm_scaled(C.t(), X, C, 1.0, 1.0)
    assert torch.equal(C, want)
