"""The kernels' gelu against 64 bits over its whole range, and on what is no number: operands that multiply to zero, so that the
bias is the argument."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# 1 (generic), tiled 256 x 256 and 128 x 128, block, skinny, ring, and the library's own choice
KERNELS = (1, 6, 17, 23, 3, 28, 0)


@pytest.mark.parametrize("kernel", KERNELS)
def test_gelu(kernel):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as hk

    tk, M, N, K = hk.tk_kernel, 32, 8192, 512
    g = torch.Generator(device="cuda").manual_seed(1)
    y = torch.cat([torch.linspace(-14, 14, N - 2048, device="cuda"), torch.randn(2048, device="cuda", generator=g)])
    special = torch.tensor([math.inf, math.nan, 0.0, -0.0, 1e30, -1e30, 3e38, -3e38, 1e-42, 7.0, -7.0, 100.0, -100.0], device="cuda")
    y[: special.numel()] = special
    A, As = hk.quantize(torch.zeros(M, K, device="cuda"))
    B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g))
    C = torch.empty(M, N, dtype=torch.float32, device="cuda")
    prev = tk.set_kernel(kernel)
    try:
        tk.dispatch_micro(A, B, As, Bs, C, bias=y, activation="gelu")
    finally:
        tk.set_kernel(prev)
    assert torch.equal(C.isnan(), C[:1].isnan().expand_as(C)) and torch.equal(C.nan_to_num(), C[:1].nan_to_num().expand_as(C))  # every row the same
    c, y = C[M - 1].double(), y.double()
    want = y * torch.special.ndtr(y)
    assert c[0] == math.inf and c[1].isnan() and (c[5] == 0) and (c[7] == 0) and c[4] == y[4] and c[6] == y[6]
    d = (c - want).abs()[2:]
    # the polynomial's 7.5e-9 of y, and of y a half ulp each of the exponent (ln 2 of it, a half at most of the result), the hardware's exp2 (one
    # ulp of at most a half), the difference from one and the product
    bound = y.abs()[2:] * (7.5e-9 + 2.0**-24 * (0.35 + 1 + 0.5 + 1)) + 1e-38
    assert (d <= bound).all(), (d / bound).max()
