"""gemm_ragged_kernel: rows that begin between two dwords, on them, or both in one operand; small integers, so that every order of summation gives
the same bits, NaN around the operands."""
import pytest
import torch

import gemm_amd as g
from gemm_amd import _abi

pytestmark = pytest.mark.gpu


# K: less than a tile, one and two with 1 to 9 elements more or less (whole tiles end eight elements before K), more tiles than are on the way;
# M, N: one row, tiles and part of one, odd and even last columns (the last chunk of a k-row begins at either)
@pytest.mark.parametrize("K", [7, 56, 64, 71, 72, 73, 128, 135, 137, 200, 263, 329, 457, 841])
@pytest.mark.parametrize("M,N", [(1, 65), (67, 130), (193, 71)])
@pytest.mark.parametrize("a_layout", [g.A_MK, g.A_KM])
@pytest.mark.parametrize("b_layout", [g.B_KN, g.B_NK])
def test_rows(M, N, K, a_layout, b_layout):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    lib, st = _abi.load(), torch.cuda.current_stream().cuda_stream or None

    def operand(rows, cols, pad, shift):
        ld = cols + pad
        buf = torch.full((shift + rows * ld + 8,), float("nan"), dtype=torch.bfloat16, device="cuda")
        m = buf[shift:shift + rows * ld].view(rows, ld)[:, :cols]
        m.copy_(torch.randint(-2, 3, (rows, cols), generator=gen, device="cuda"))
        return m, ld

    for pad, shift in ((0, 0), (1, 0), (2, 1), (3, 2), (8 - K % 8, 1)):
        (A, lda), (B, ldb) = operand(*((M, K) if a_layout == g.A_MK else (K, M)), pad, shift), operand(*((K, N) if b_layout == g.B_KN else (N, K)), pad ^ 1, shift)
        want = ((A if a_layout == g.A_MK else A.t()).float() @ (B if b_layout == g.B_KN else B.t()).float()).to(torch.bfloat16)
        for c_layout in (g.C_ROW, g.C_COL):
            C = torch.full((M, N) if c_layout == g.C_ROW else (N, M), float("nan"), dtype=torch.bfloat16, device="cuda")
            args = (A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, lda, ldb, C.stride(0))
            if M * K >= 8 and _abi.call_kernel(*args, b_layout, c_layout, a_layout, ws_bytes=0) != "ragged":
                assert (pad, shift, M) != (2, 1, 67)
                continue
            assert lib.neogemm_bf16_general(*args, a_layout, b_layout, c_layout, 1.0, 0.0, 0, 0, 0, 1, None, 0, st) == _abi.OK
            assert torch.equal(C if c_layout == g.C_ROW else C.t(), want), (pad, shift, c_layout)


def test_fewer_splits_than_planned():
    """A workspace for some of the planned splits: as many as it holds."""
    M, N, K = 67, 1081, 4253
    gen = torch.Generator(device="cuda").manual_seed(1)
    A, B = (torch.randint(-1, 2, s, generator=gen, device="cuda").to(torch.bfloat16) for s in ((M, K), (K, N)))
    want = (A.float() @ B.float()).to(torch.bfloat16)
    need = _abi.call_workspace_bytes(A.data_ptr(), B.data_ptr(), M, N, K, K, N, g.B_KN, g.C_ROW)
    assert need >= 3 * M * N * 4
    ws = torch.full((need // 4 + 4,), float("nan"), device="cuda")
    for size in (need, need - 4, 2 * M * N * 4, M * N * 4, 0):
        ws.fill_(float("nan"))
        C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert _abi.load().neogemm_bf16_general(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K, N, N, g.A_MK, g.B_KN, g.C_ROW, 1.0, 0.0, 0, 0, 0, 1,
                                                ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream or None) == _abi.OK
        assert torch.equal(C, want)
        assert bool(torch.isnan(ws[size // 4:]).all())
