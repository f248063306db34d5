"""The tile kernels' stores of whole lines against the one-wave-per-tile kernel, bit for bit (every kernel adds K in the same order): rows
on both sides of the 8, 16 and 32 that a store covers, columns that end inside a line, bf16 and fp32, and what lies around C."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as m

    return m


@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N", [(1, 8), (7, 72), (8, 64), (9, 40), (17, 136), (136, 264), (263, 520), (512, 1032)])
def test_line_stores(hk, M, N, out):
    tk, K, pad = hk.tk_kernel, 384, 4096
    g = torch.Generator(device="cuda").manual_seed(M * N)
    A, As = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
    B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g))
    want = None
    # 1: one wave per tile; 2: tiled; 5, 6, 17: its tiles of 128 x 256, 256 x 256, 128 x 128; 23, 24, 26: block
    for kernel in (1, 2, 5, 6, 17, 23, 24, 26):
        whole = torch.full((2 * pad + M * N,), 7.0, dtype=out, device="cuda")
        C = whole[pad : pad + M * N].view(M, N)
        prev, prev_split = tk.set_kernel(kernel), tk.set_k_split(1)
        try:
            tk.dispatch_micro(A, B, As, Bs, C)
        finally:
            tk.set_kernel(prev)
            tk.set_k_split(prev_split)
        assert (whole[:pad] == 7).all() and (whole[pad + M * N :] == 7).all(), kernel
        want = C.clone() if want is None else want
        assert torch.equal(C, want), kernel


@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(300, 6001, 1056), (1001, 3003, 1056)])
def test_line_stores_of_ragged_products(hk, M, N, K, out):
    """Rows that start at any element: the block kernel's ragged instantiation, which the library takes
    here, stores runs of 16 bytes or, across N, elements."""
    tk, pad = hk.tk_kernel, 4096
    g = torch.Generator(device="cuda").manual_seed(M * N)
    A, As = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
    B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g))
    res = []
    for kernel in (1, 0):
        whole = torch.full((2 * pad + M * N,), 7.0, dtype=out, device="cuda")
        C = whole[pad : pad + M * N].view(M, N)
        prev, prev_split = tk.set_kernel(kernel), tk.set_k_split(1)
        try:
            tk.dispatch_micro(A, B, As, Bs, C)
        finally:
            tk.set_kernel(prev)
            tk.set_k_split(prev_split)
        assert (whole[:pad] == 7).all() and (whole[pad + M * N :] == 7).all(), kernel
        res.append(C)
    assert torch.equal(*res)
