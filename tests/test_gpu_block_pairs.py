"""The block kernel's ring of two-K-tile chunks (kernel 24) against its ring of single K-tiles (kernel 23), bit for bit -- both add
K in the same order -- at odd and even numbers of K-tiles, with fewer chunks than slots, at tile edges, in every pair of layouts.
(Kernel 23 itself is held to the oracle in test_gpu_parity.py.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as m

    return m


@pytest.mark.parametrize("K", [128, 256, 384, 512, 640, 768, 896, 1152, 1664, 2176])
@pytest.mark.parametrize("M,N", [(1, 8), (96, 160), (128, 128), (161, 264), (320, 416)])
def test_pairs_match_single_k_tiles(hk, M, N, K):
    tk = hk.tk_kernel
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, As = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
    B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g), 3)
    for la in (0, 1) if M % 32 == 0 else (0,):
        for lb in (0, 1) if N % 32 == 0 else (0,):
            a = (hk.tile_operand(A), hk.tile_scales(As, K)) if la else (A, As)
            b = (hk.tile_operand(B), hk.tile_scales(Bs, K)) if lb else (B, Bs)
            out = []
            for kernel in (23, 24):
                C = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
                prev = tk.set_kernel(kernel)
                try:
                    tk.dispatch_micro(a[0], b[0], a[1], b[1], C, 2, 3, la, lb)
                finally:
                    tk.set_kernel(prev)
                out.append(C)
            assert torch.isfinite(out[0]).all() and torch.equal(*out), (la, lb)
