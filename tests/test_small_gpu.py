"""Small problems (64x64 and 128x64 tiles of gemm_roles_kernel): small integers, so that every order of summation gives the same bits."""
import pytest
import torch

import gemm_amd as g
from gemm_amd import _abi

pytestmark = pytest.mark.gpu


# K: part of a stage, one, two, three (the ring's depth), four, a partial last one, split; M, N: edges of the 64 tile, one column of chunks,
# up to one 64x64 tile per CU, and more
@pytest.mark.parametrize("M,N,K", [(136, 136, 8), (136, 8, 64), (264, 200, 72), (328, 448, 128), (448, 448, 184), (192, 520, 256), (640, 640, 640), (1024, 1024, 1024),
                                   (1152, 1152, 320), (1024, 2048, 264), (264, 264, 4104), (256, 256, 8192), (256, 1024, 1024)])
@pytest.mark.parametrize("a_layout", [g.A_MK, g.A_KM])
@pytest.mark.parametrize("b_layout", [g.B_KN, g.B_NK])
@pytest.mark.parametrize("c_layout", [g.C_ROW, g.C_COL])
def test_small(M, N, K, a_layout, b_layout, c_layout):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)

    def ints(rows, cols, pad):   # NaN between the rows
        m = torch.full((rows, cols + pad), float("nan"), dtype=torch.bfloat16, device="cuda")
        m[:, :cols] = torch.randint(-2, 3, (rows, cols), generator=gen, device="cuda")
        return m[:, :cols]

    A, B = ints(*((M, K) if a_layout == g.A_MK else (K, M)), 8), ints(*((K, N) if b_layout == g.B_KN else (N, K)), 16)
    want = (A if a_layout == g.A_MK else A.t()).float() @ (B if b_layout == g.B_KN else B.t()).float()
    # (324 and 512 tiles of 64x64 are more than CUs: 180 and 256 of 128x64 instead)
    kernel = "roles 128x64" if (M, N, K) in ((1152, 1152, 320), (1024, 2048, 264)) else "roles 64x64"
    C = torch.full((M, N) if c_layout == g.C_ROW else (N, M), float("nan"), dtype=torch.bfloat16, device="cuda")
    got = C if c_layout == g.C_ROW else C.t()
    assert _abi.call_kernel(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0), B.stride(0), C.stride(0), b_layout, c_layout,
                            a_layout) == kernel
    g.gemm_into(A, B, C, M, N, K, A.stride(0), B.stride(0), C.stride(0), b_layout, c_layout, a_layout=a_layout)
    assert torch.equal(got, want.to(torch.bfloat16))
    old = got.clone()
    g.gemm_into(A, B, C, M, N, K, A.stride(0), B.stride(0), C.stride(0), b_layout, c_layout, a_layout=a_layout, alpha=0.5, beta=-1.0)
    assert torch.equal(got, (0.5 * want - old.float()).to(torch.bfloat16))
