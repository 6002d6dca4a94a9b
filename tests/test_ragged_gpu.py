"""Operands at any address and with any leading dimension (gemm_ragged_kernel): small integers between NaNs, so that every order
of summation gives the same bits and an element that does not belong to the product shows."""
import pytest
import torch

import gemm_amd as g
import neoGEMM
from gemm_amd import _abi

pytestmark = pytest.mark.gpu


def between_nans(gen, rows, cols, pad, shift):
    """A rows x cols matrix of small integers, its rows cols + pad apart, `shift` elements into a buffer that is NaN elsewhere."""
    ld = cols + pad
    flat = torch.full((rows * ld + shift + 3,), float("nan"), dtype=torch.bfloat16, device="cuda")
    m = flat[shift:shift + rows * ld].view(rows, ld)[:, :cols]
    m.copy_(torch.randint(-2, 3, (rows, cols), generator=gen, device="cuda"))
    return m


# K: one element, less than a chunk, around one, two, three and five tiles of 64 (prologue, plain loop, careful tail), deep enough to
# be split; M, N: one row, less than a chunk, edges of the 64 and 128 tiles, enough tiles for the 128 one
SIZES = [(9, 9, 1), (1, 9, 13), (17, 1, 9), (64, 65, 7), (63, 129, 64), (65, 64, 71), (130, 127, 129), (129, 257, 193), (65, 191, 322), (200, 77, 447),
         (1, 1001, 1537), (127, 131, 4099), (2500, 2501, 137), (3001, 2999, 520)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("a_layout", [g.A_MK, g.A_KM])
@pytest.mark.parametrize("b_layout", [g.B_KN, g.B_NK])
@pytest.mark.parametrize("c_layout", [g.C_ROW, g.C_COL])
def test_operands_at_any_address(M, N, K, a_layout, b_layout, c_layout):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    for pad_a, pad_b, shift in ((0, 1, 1), (3, 0, 2)):
        A = between_nans(gen, *((M, K) if a_layout == g.A_MK else (K, M)), pad_a, shift)
        B = between_nans(gen, *((K, N) if b_layout == g.B_KN else (N, K)), pad_b, shift + 1)
        At, Bkn = A if a_layout == g.A_MK else A.t(), B if b_layout == g.B_KN else B.t()
        want = At.float() @ Bkn.float()
        C = torch.full((M, N) if c_layout == g.C_ROW else (N, M), float("nan"), dtype=torch.bfloat16, device="cuda")
        g.gemm_into(A, B, C, M, N, K, A.stride(0), B.stride(0), C.stride(0), b_layout, c_layout, a_layout=a_layout)
        got = C if c_layout == g.C_ROW else C.t()
        assert torch.equal(got, want.to(torch.bfloat16))
        old = got.clone()
        g.gemm_into(A, B, C, M, N, K, A.stride(0), B.stride(0), C.stride(0), b_layout, c_layout, a_layout=a_layout, alpha=0.5, beta=-1.0)
        assert torch.equal(got, (0.5 * want - old.float()).to(torch.bfloat16))


def test_the_last_bytes_of_an_allocation():
    """Operands that end where their buffer of a few elements ends."""
    for M, N, K in ((1, 1, 8), (2, 3, 5), (3, 2, 7), (1, 8, 1), (8, 1, 1)):
        A, B = torch.ones(M, K, dtype=torch.bfloat16, device="cuda"), torch.ones(K, N, dtype=torch.bfloat16, device="cuda")
        assert torch.equal(neoGEMM.gemm(A, B), torch.full((M, N), float(K), dtype=torch.bfloat16, device="cuda"))


def test_split_needs_the_general_call_and_its_workspace():
    """K is split over the workspace the query asks for; with less, and through the calls that never took one, it is not."""
    M, N, K = 127, 131, 8191
    gen = torch.Generator(device="cuda").manual_seed(7)
    A, B = between_nans(gen, M, K, 0, 1), between_nans(gen, K, N, 0, 1)
    want = (A.float() @ B.float()).to(torch.bfloat16)
    lib = _abi.load()
    need = int(lib.neogemm_bf16_call_workspace_bytes(A.data_ptr(), B.data_ptr(), M, N, K, K, N, g.A_MK, g.B_KN, g.C_ROW, 0, 0, 1))
    assert need >= 2 * M * N * 4
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    st = torch.cuda.current_stream().cuda_stream or None
    for size in (need, need - 1, 0):
        C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert lib.neogemm_bf16_general(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K, N, N, g.A_MK, g.B_KN, g.C_ROW, 1.0, 0.0, 0, 0, 0, 1,
                                        ws.data_ptr(), size, st) == _abi.OK
        assert torch.equal(C, want)
    C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert lib.neogemm_bf16(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K, N, N, g.B_KN, g.C_ROW, None, 0, st) == _abi.OK
    assert torch.equal(C, want)


# batches: transposed views, slices of a larger tensor, a shared operand, odd sizes; K of one and two tiles
@pytest.mark.parametrize("b,M,N,K", [(3, 200, 136, 64), (2, 264, 392, 128), (5, 77, 77, 96), (3, 100, 64, 101), (1, 96, 520, 72), (4, 1, 9, 200), (2, 9, 1, 5)])
def test_batches_of_views(b, M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(b + M)

    def ints(*shape):
        return torch.randint(-2, 3, shape, generator=gen, device="cuda").to(torch.bfloat16)

    As = [ints(b, M, K), ints(b, K, M).transpose(1, 2), ints(b, M, K + 5)[:, :, 3:K + 3], ints(M, b, K).transpose(0, 1), ints(1, M, K).expand(b, M, K),
          ints(K, b, M).permute(1, 2, 0)]
    Bs = [ints(b, K, N), ints(b, N, K).transpose(1, 2), ints(K, N), ints(N, K).t(), ints(b, K + 1, N)[:, 1:], ints(K, N, b).permute(2, 0, 1)]
    for A in As:
        for B in Bs:
            want = torch.stack([A[i].float() @ (B[i] if B.dim() == 3 else B).float() for i in range(b)])
            assert torch.equal(neoGEMM.bmm(A, B), want.to(torch.bfloat16))


# large enough that copies on the 16-byte grid pay: K a part of a chunk past a tile, MN-major rows that end inside a chunk, one operand
# on the grid already, K split, a batch with a shared and with a strided operand
@pytest.mark.parametrize("b,M,N,K", [(1, 2501, 2503, 2505), (1, 603, 1584, 15177), (1, 4097, 3080, 3001), (1, 3501, 2001, 2000), (3, 2001, 2003, 2005)])
def test_copies_on_the_grid(b, M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    lib = _abi.load()
    st = torch.cuda.current_stream().cuda_stream or None
    for a_layout in (g.A_MK, g.A_KM):
        for b_layout in (g.B_KN, g.B_NK):
            for c_layout in (g.C_ROW, g.C_COL):
                A = between_nans(gen, *((b * M, K) if a_layout == g.A_MK else (b * K, M)), 0, 1)
                B = between_nans(gen, *((K, N) if b_layout == g.B_KN else (N, K)), 0, 8)
                A3 = A.view(b, -1, A.shape[1])
                want = (A3 if a_layout == g.A_MK else A3.transpose(1, 2)).float() @ (B if b_layout == g.B_KN else B.t()).float()
                old = torch.randint(-8, 9, (b, M, N) if c_layout == g.C_ROW else (b, N, M), generator=gen, device="cuda").to(torch.bfloat16)
                C = old.clone()
                lda, ldb, sa = A.stride(0), B.stride(0), A3.stride(0) if b > 1 else 0
                need = int(lib.neogemm_bf16_call_workspace_bytes(A.data_ptr(), B.data_ptr(), M, N, K, lda, ldb, a_layout, b_layout, c_layout, sa, 0, b))
                ws = torch.full((need // 4 + 4,), float("nan"), device="cuda")
                for size in (need, 0):   # with the copies, and by the kernel that reads in place
                    kernel = _abi.call_kernel(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, lda, ldb, C.stride(1), b_layout, c_layout, a_layout, 1.0,
                                              sa, 0, M * N, b, size)
                    assert kernel.startswith("copy+") if size else kernel == "ragged"
                    C.copy_(old)
                    assert lib.neogemm_bf16_general(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, lda, ldb, C.stride(1), a_layout, b_layout, c_layout,
                                                    1.0, 1.0, sa, 0, M * N, b, ws.data_ptr(), size, st) == _abi.OK
                    got, add = (C, old) if c_layout == g.C_ROW else (C.transpose(1, 2), old.transpose(1, 2))
                    assert torch.equal(got, (want + add.float()).to(torch.bfloat16))


# few rows of A off the grid beside a B on it: copies of A alone for the decode kernels, every number of row fragments, K whose last
# chunk is part padding (B [K,N]; the k-rows behind K are NaN), K split
@pytest.mark.parametrize("M,N,K,b_layout,kernel", [
    (5, 4104, 1025, g.B_KN, "skinny"), (16, 12296, 6001, g.B_KN, "skinny"), (20, 6152, 2001, g.B_KN, "skinny"), (33, 13144, 20789, g.B_KN, "skinny"),
    (70, 13872, 4142, g.B_KN, "skinny"), (92, 15272, 5205, g.B_KN, "skinny"), (50, 5752, 6945, g.B_KN, "strip"), (63, 5552, 13379, g.B_KN, "strip"),
    (16, 2056, 1024, g.B_NK, "skinny"), (32, 1032, 1024, g.B_NK, "skinny"), (33, 13376, 14376, g.B_NK, "skinny"), (72, 14344, 7840, g.B_NK, "skinny"),
    (96, 14344, 4096, g.B_NK, "skinny"), (104, 4104, 4096, g.B_NK, "strip"), (128, 4104, 4096, g.B_NK, "strip"), (72, 6648, 8896, g.B_NK, "strip")])
@pytest.mark.parametrize("c_layout", [g.C_ROW, g.C_COL])
def test_copies_for_the_decode_kernels(M, N, K, b_layout, kernel, c_layout):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = between_nans(gen, M, K, 0, 1), between_nans(gen, *((K, N) if b_layout == g.B_KN else (N, K)), 8, 8)
    want = A.float() @ (B if b_layout == g.B_KN else B.t()).float()
    C = torch.full((M, N) if c_layout == g.C_ROW else (N, M), float("nan"), dtype=torch.bfloat16, device="cuda")
    got = C if c_layout == g.C_ROW else C.t()
    assert _abi.call_kernel(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K, B.stride(0), C.stride(0), b_layout, c_layout) == "copy+" + kernel
    g.gemm_into(A, B, C, M, N, K, K, B.stride(0), C.stride(0), b_layout, c_layout)
    assert torch.equal(got, want.to(torch.bfloat16))
    old = got.clone()
    g.gemm_into(A, B, C, M, N, K, K, B.stride(0), C.stride(0), b_layout, c_layout, alpha=0.5, beta=-1.0)
    assert torch.equal(got, (0.5 * want - old.float()).to(torch.bfloat16))


# copies of more than 256 MiB in panels: of the rows, of the columns, of both (a panel of A copied for each panel of columns), of the
# problems of a batch; a last panel of one row, split otherwise than the others; rows of A [K,M] 2^21 elements apart and more
@pytest.mark.parametrize("b,M,N,K,a_layout,b_layout,c_layout", [
    (1, 70001, 2056, 2049, g.A_MK, g.B_KN, g.C_ROW), (1, 70001, 2056, 2048, g.A_KM, g.B_KN, g.C_COL), (1, 513, 70003, 2049, g.A_MK, g.B_NK, g.C_ROW),
    (1, 4001, 4001, 40001, g.A_MK, g.B_KN, g.C_COL), (1, 4001, 4003, 40001, g.A_KM, g.B_NK, g.C_ROW), (1, 513, 4104, 300001, g.A_MK, g.B_KN, g.C_ROW),
    (41, 1501, 1503, 1801, g.A_MK, g.B_KN, g.C_ROW), (1, 2097167, 264, 16, g.A_KM, g.B_KN, g.C_ROW)])
def test_copies_in_panels(b, M, N, K, a_layout, b_layout, c_layout):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)

    def ints(*shape):
        return torch.randint(-2, 3, shape, generator=gen, device="cuda", dtype=torch.int8).to(torch.bfloat16)

    A, B = ints(b, *((M, K) if a_layout == g.A_MK else (K, M))), ints(b, *((K, N) if b_layout == g.B_KN else (N, K)))
    C = ints(b, *((M, N) if c_layout == g.C_ROW else (N, M)))
    old, got = C.clone(), C if c_layout == g.C_ROW else C.transpose(1, 2)
    strides = (A.stride(0), B.stride(0)) if b > 1 else (0, 0)
    need = _abi.call_workspace_bytes(A.data_ptr(), B.data_ptr(), M, N, K, A.stride(1), B.stride(1), b_layout, c_layout, a_layout, *strides, b)
    ws = torch.full((need // 4 + 4,), float("nan"), device="cuda")
    assert _abi.call_kernel(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(1), B.stride(1), C.stride(1), b_layout, c_layout, a_layout, 1.0,
                            *strides, M * N, b, need).startswith("copy+")
    assert A.numel() * 2 + (B.numel() * 2 if B.stride(1) % 8 else 0) > 256 << 20 or A.stride(1) >= 1 << 21
    assert _abi.load().neogemm_bf16_general(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(1), B.stride(1), C.stride(1), a_layout, b_layout,
                                            c_layout, 1.0, 1.0, *strides, M * N, b, ws.data_ptr(), need,
                                            torch.cuda.current_stream().cuda_stream or None) == _abi.OK
    assert bool(torch.isnan(ws[need // 4:]).all())
    for i in range(b):
        want = (A[i] if a_layout == g.A_MK else A[i].t()).float() @ (B[i] if b_layout == g.B_KN else B[i].t()).float()
        want += (old[i] if c_layout == g.C_ROW else old[i].t()).float()
        assert torch.equal(got[i], want.to(torch.bfloat16))


# K of at most 128 with both operands K-major and enough tiles: one and two 64-deep units, whole and partial; rows and columns that end
# inside a block, a run of column tiles per workgroup that does not divide them, C at odd addresses, alpha
@pytest.mark.parametrize("b,M,N,K", [(32, 1024, 1024, 128), (40, 517, 801, 96), (1, 4100, 3001, 64), (7, 2048, 1000, 8), (300, 129, 129, 72), (1, 130, 60000, 104),
                                     (1, 70000, 70, 120)])
@pytest.mark.parametrize("c_layout", [g.C_ROW, g.C_COL])
def test_short_k(b, M, N, K, c_layout):
    gen = torch.Generator(device="cuda").manual_seed(b + M + N + K)

    def ints(*shape):
        return torch.randint(-2, 3, shape, generator=gen, device="cuda").to(torch.bfloat16)

    A, B = ints(b, M, K + 8), ints(b, N, K)
    want = 0.5 * (A[:, :, :K].float() @ B.transpose(1, 2).float())
    A[:, :, K:] = float("nan")
    C = torch.full((b, M, N) if c_layout == g.C_ROW else (b, N, M), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert _abi.call_kernel(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K + 8, K, C.stride(1), g.B_NK, c_layout, stride_a=M * (K + 8),
                            stride_b=N * K, stride_c=M * N, batch=b) == "short K"
    assert _abi.load().neogemm_bf16_general(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K + 8, K, C.stride(1), g.A_MK, g.B_NK, c_layout, 0.5, 0.0,
                                            M * (K + 8), N * K, M * N, b, None, 0, torch.cuda.current_stream().cuda_stream or None) == _abi.OK
    assert torch.equal(C if c_layout == g.C_ROW else C.transpose(1, 2), want.to(torch.bfloat16))
