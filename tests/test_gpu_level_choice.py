"""The ring kernel and the block kernel's K split where the two are level, and next to it: the automatic call runs one of them (as the route
says) and gives its bits, and it is no slower than the better one by more than two calibrations of one point differ."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(28, 3584, 15360), (36, 6656, 13312), (64, 3584, 15360), (65, 3584, 15360), (64, 8192, 28672)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("tile_b", [0, 1])
def test_automatic_call_is_either_kernel(route, M, N, K, tile_b):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as hk

    tk = hk.tk_kernel
    g = torch.Generator(device="cuda").manual_seed(M)
    A, As = hk.quantize(torch.randn(M, K, device="cuda", generator=g), 2)
    B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g).mul_(0.02), 2)
    if tile_b:
        B, Bs = hk.tile_operand(B), hk.tile_scales(Bs, K)
    got = torch.full((M, N), float("nan"), device="cuda")
    taken = route.gemm(A, B, As, Bs, got, M, N, K, lb=tile_b)
    assert taken & (0xFF | route.SPLIT) in (route.RING, route.RING | route.SPLIT, route.BLOCK | route.SPLIT), hex(taken)
    kernel, split = (28, 0) if taken & 0xFF == route.RING else (22, -1)
    code = tk.kernel_choice(M, N, K, 0, tile_b)
    assert code == (28 if kernel == 28 else 27)
    want = torch.full((M, N), float("nan"), device="cuda")
    prev = tk.set_kernel(kernel), tk.set_k_split(split)
    try:
        tk.dispatch_micro(A, B, As, Bs, want, 2, 2, 0, tile_b)
    finally:
        tk.set_kernel(prev[0]), tk.set_k_split(prev[1])
    assert torch.equal(got, want)
