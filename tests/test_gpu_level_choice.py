"""The ring kernel against the block kernel's K split where the choice takes the two as level, and next to it: what the automatic call
takes is one of the two, and agrees with both within what the order of the sum may change."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(28, 3584, 15360), (36, 6656, 13312), (64, 3584, 15360), (65, 3584, 15360)])
@pytest.mark.parametrize("tile_b", [0, 1])
def test_automatic_call_is_either_kernel(M, N, K, tile_b):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as hk
    from oracle import c_oracle

    tk = hk.tk_kernel
    g = torch.Generator(device="cuda").manual_seed(M)
    A, As = hk.quantize(torch.randn(M, K, device="cuda", generator=g), 2)
    B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g).mul_(0.02), 2)
    a, b = (torch.from_numpy(c_oracle.dequantise(q.cpu().numpy(), s.cpu().numpy(), 2)).cuda().abs() for q, s in ((A, As), (B, Bs)))
    size = a @ b.T  # the sum of the terms' sizes
    if tile_b:
        B, Bs = hk.tile_operand(B), hk.tile_scales(Bs, K)
    res = []
    for kernel in (0, 28, 24):
        C = torch.full((M, N), float("nan"), device="cuda")
        prev = tk.set_kernel(kernel)
        try:
            tk.dispatch_micro(A, B, As, Bs, C, 2, 2, 0, tile_b)
        finally:
            tk.set_kernel(prev)
        res.append(C)
    # the products are exact; each of the two sums rounds once per 64 values of K and once per share
    bound = 2 * (K // 64 + 16) * 2.0**-24 * size
    for other in res[1:]:
        assert ((res[0] - other).abs() <= bound).all()
