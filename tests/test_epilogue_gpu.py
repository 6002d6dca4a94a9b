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
