"""C = alpha * A*B + beta * C through the staged epilogue of every tile kernel: small integers, so that the result does not
depend on the order of the sums and is compared bit for bit with the fp32 expression rounded once."""
import pytest
import torch

import gemm_amd as g

pytestmark = pytest.mark.gpu


def small_ints(gen, *shape, top=2):
    return torch.randint(-top, top + 1, shape, generator=gen, device="cuda").to(torch.bfloat16)


# (M, N, K, ldc - N, kernel): whole and ragged tiles, a last column group that is not whole (ldc padded to 8), column-major C
@pytest.mark.parametrize("M,N,K,pad,variant", [
    (512, 768, 256, 0, g.VARIANT_T64x64_W4), (300, 520, 200, 0, g.VARIANT_T64x64_W4), (1000, 1028, 512, 4, g.VARIANT_T64x128_W4),
    (2568, 2056, 512, 0, g.VARIANT_T128x128_W4), (3077, 3080, 256, 0, g.VARIANT_T192x256_W4), (5128, 5124, 256, 4, g.VARIANT_C256x256_W4),
    (5128, 5128, 264, 0, g.VARIANT_T256x256_W4)])
@pytest.mark.parametrize("c_layout", [g.C_ROW, g.C_COL])
def test_accumulating_epilogue(M, N, K, pad, variant, c_layout):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = small_ints(gen, M, K), small_ints(gen, N, K)
    if c_layout == g.C_COL:   # the kernels see the transposed problem: M is what C's rows hold in memory
        A, B = B, A
        M, N = N, M
    assert g.plan(M, N, K, g.B_NK, c_layout)[0] == variant
    rows, cols = (M, N) if c_layout == g.C_ROW else (N, M)
    buf = small_ints(gen, rows, cols + pad, top=8)
    want = buf.clone()
    prod = A.float() @ B.float().t()
    want[:, :cols] = (0.5 * (prod if c_layout == g.C_ROW else prod.t()) - 3.0 * buf[:, :cols].float()).to(torch.bfloat16)
    g.gemm_into(A, B, buf, M, N, K, K, K, cols + pad, g.B_NK, c_layout, alpha=0.5, beta=-3.0)
    assert torch.equal(buf, want)   # the padding between rows included


# C at any element and with any leading dimension: staged stores of the tile kernels, strips, the skinny kernel, the fp32 partials
# of a split and their reduction (rows of partials that straddle a lane's four elements), each to the edge of an odd N
@pytest.mark.parametrize("M,N,K", [(300, 521, 200), (5128, 5125, 256), (1000, 1027, 512), (16, 1001, 4096), (3, 4099, 1024), (128, 4097, 16384),
                                   (120, 14339, 2048), (256, 261, 8192), (257, 131, 16384)])
@pytest.mark.parametrize("c_layout", [g.C_ROW, g.C_COL])
@pytest.mark.parametrize("shift", [1, 2])
def test_c_at_any_address(M, N, K, c_layout, shift):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = small_ints(gen, M, K, top=1), small_ints(gen, N, K, top=1)
    rows, cols = (M, N) if c_layout == g.C_ROW else (N, M)
    ldc = cols + shift
    flat = small_ints(gen, rows * ldc + shift, top=8)
    want = flat.clone()
    prod = A.float() @ B.float().t()
    prod = prod if c_layout == g.C_ROW else prod.t()
    view = want[shift:].view(rows, ldc)[:, :cols]
    old = view.clone()
    view.copy_(prod.to(torch.bfloat16))
    C = flat.clone()
    g.gemm_into(A, B, C[shift:], M, N, K, K, K, ldc, g.B_NK, c_layout)
    assert torch.equal(C, want)   # what lies between the rows included
    C = flat.clone()
    view.copy_((2.0 * prod + old.float()).to(torch.bfloat16))
    g.gemm_into(A, B, C[shift:], M, N, K, K, K, ldc, g.B_NK, c_layout, alpha=2.0, beta=1.0)
    assert torch.equal(C, want)


def test_odd_c_without_a_workspace():
    """A shape whose plan splits K, into a C on odd addresses, with no workspace: unsplit, as such a C always ran."""
    from gemm_amd import _abi
    M, N, K = 256, 261, 8192
    gen = torch.Generator(device="cuda").manual_seed(1)
    A, B = small_ints(gen, M, K, top=1), small_ints(gen, N, K, top=1)
    C = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    assert g.plan(M, N, K, g.B_NK)[1] > 1
    st = _abi.gemm_raw(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K, K, N, g.B_NK, g.C_ROW, 0, 0, torch.cuda.current_stream().cuda_stream)
    assert st == _abi.OK and torch.equal(C, (A.float() @ B.float().t()).to(torch.bfloat16))


@pytest.mark.parametrize("c_layout", [g.C_ROW, g.C_COL])
def test_odd_c_stride_without_a_workspace(c_layout):
    """The same for the problems of a batch, whose outputs lie an odd number of elements apart."""
    from gemm_amd import _abi
    b, M, N, K = 2, 64, 64, 8192
    gen = torch.Generator(device="cuda").manual_seed(2)
    A, B = small_ints(gen, b, M, K, top=1), small_ints(gen, b, N, K, top=1)
    lib = _abi.load()
    assert lib.neogemm_bf16_batched_workspace_bytes(M, N, K, b) > 0
    flat = torch.full((b * (M * N + 1),), 5.0, dtype=torch.bfloat16, device="cuda")
    st = lib.neogemm_bf16_batched(A.data_ptr(), B.data_ptr(), flat.data_ptr(), M, N, K, K, K, N, M * K, N * K, M * N + 1, b, g.B_NK, c_layout,
                                  None, 0, torch.cuda.current_stream().cuda_stream or None)
    assert st == _abi.OK
    want = torch.stack([A[i].float() @ B[i].float().t() for i in range(b)])
    want = (want if c_layout == g.C_ROW else want.transpose(1, 2)).reshape(b, M * N).to(torch.bfloat16)
    assert torch.equal(flat.view(b, M * N + 1)[:, :M * N], want) and bool((flat.view(b, M * N + 1)[:, M * N] == 5.0).all())
