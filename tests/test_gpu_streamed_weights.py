"""Weights of 128 MB and more, which the tiled kernel's K split and the block kernel read with the non-temporal bit where they are tile-major and
one tile row meets them: the same rows with a second tile row behind them, which are read without it, give the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def operands():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as hk

    made = {}

    def get(N, K):
        if (N, K) not in made:
            made.clear()
            g = torch.Generator(device="cuda").manual_seed(N)
            B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g).mul_(0.02), 2)
            made[N, K] = hk, hk.quantize(torch.randn(512, K, device="cuda", generator=g), 2), (B, Bs), (hk.tile_operand(B), hk.tile_scales(Bs, K))
            assert B.numel() >= 128 << 20
        return made[N, K]

    return get


# kernel, rows of one tile row, shares of K (1: unsplit), N, K
@pytest.mark.parametrize("kernel,rows,shares,N,K", [(6, 256, 4, 8192, 22528), (5, 128, 2, 8192, 22528), (24, 128, 2, 8192, 22528), (24, 128, 3, 5120, 35200), (24, 128, 1, 24576, 7680)])
@pytest.mark.parametrize("tile_b", [0, 1])
@pytest.mark.parametrize("out,act", [(torch.bfloat16, None), (torch.bfloat16, "silu"), (torch.float32, None)])
def test_one_tile_row_matches_two(operands, route, kernel, rows, shares, N, K, tile_b, out, act):
    hk, (A, As), row, tile = operands(N, K)
    B, Bs = tile if tile_b else row
    tk, res = hk.tk_kernel, []
    for M in (rows, rows - 3, 2 * rows):
        C = torch.full((M, N), float("nan"), dtype=out, device="cuda")
        prev, prev_split = tk.set_kernel(kernel), tk.set_k_split(shares)
        try:
            tk.dispatch_micro(A[:M], B, As[:M], Bs, C, 2, 2, 0, tile_b, activation=act)
        finally:
            tk.set_kernel(prev)
            tk.set_k_split(prev_split)
        res.append(C)
        if act is None:
            route.gemm(A[:M], B, As[:M], Bs, torch.empty_like(C), M, N, K, lb=tile_b, kernel=kernel, k_split=shares)
            assert bool(route.memory & route.STREAM_B) == (tile_b == 1 and M <= rows)
    assert torch.isfinite(res[2]).all() and torch.equal(res[0], res[2][:rows]) and torch.equal(res[1], res[2][: rows - 3])
