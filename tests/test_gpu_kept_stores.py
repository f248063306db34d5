"""C goes out non-temporally or through the L2s by its size, row pitch and address: both ways give the same bits, on both sides of the line."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LIMIT = 16 << 20  # bytes of C whose rows start inside lines


# kernel (0: the block kernel's ragged instantiation), N, K, rows past a multiple of the tile
@pytest.mark.parametrize("kernel,N,K,rem", [(2, 4104, 256, 0), (2, 4104, 256, 9), (5, 4104, 256, 5), (6, 4168, 256, 3), (22, 4104, 256, 1), (22, 4168, 1152, 0), (24, 4104, 256, 0), (0, 4107, 1056, 0), (0, 4099, 2080, 7)])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_large_output_matches_its_parts(kernel, N, K, rem, out):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as hk

    tk, size = hk.tk_kernel, torch.finfo(out).bits // 8
    limit = (32 << 20) if kernel == 0 and size == 2 else LIMIT
    step = 512
    M = (limit // (N * size) // step + 2) * step + rem  # past the line; its parts of `step` rows are below
    assert (N * size) % 128 and M * N * size > limit and step * N * size < limit
    g = torch.Generator(device="cuda").manual_seed(N)
    A, As = hk.quantize(torch.randn(M, K, device="cuda", generator=g), 2)
    B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g).mul_(0.05), 2)
    guard = torch.full((M * N + 512,), 7.0, dtype=out, device="cuda")
    prev, prev_split = tk.set_kernel(kernel), tk.set_k_split(1)
    try:
        C = guard[256 : 256 + M * N].view(M, N)
        tk.dispatch_micro(A, B, As, Bs, C, 2, 2)
        for m in range(0, M, step):
            part = torch.full((min(step, M - m), N), float("nan"), dtype=out, device="cuda")
            tk.dispatch_micro(A[m : m + step], B, As[m : m + step], Bs, part, 2, 2)
            assert torch.equal(part, C[m : m + step]), m
    finally:
        tk.set_kernel(prev)
        tk.set_k_split(prev_split)
    assert (guard[:256] == 7).all() and (guard[256 + M * N :] == 7).all()


# on both sides of each line of the rule: up to 64 rows; 4 MB of C; bf16 32 MB, fp32 never non-temporally, but rows and an address that start on lines
@pytest.mark.parametrize("M,N,K,out,shift,form", [
    (64, 20001, 1056, torch.float32, 0, "PIECES"), (65, 20001, 1056, torch.float32, 0, "KEPT"), (65, 16001, 1056, torch.float32, 0, "PIECES"),
    (300, 6989, 1056, torch.bfloat16, 0, "PIECES"), (300, 7001, 1056, torch.bfloat16, 0, "OUT"), (2100, 7989, 1056, torch.bfloat16, 0, "OUT"),
    (2100, 7991, 1056, torch.bfloat16, 0, "KEPT"), (1100, 1024, 1056, torch.float32, 0, "OUT"), (1100, 1024, 1056, torch.float32, 1, "KEPT"),
    (2100, 8000, 1056, torch.bfloat16, 0, "OUT"), (2100, 8000, 1056, torch.bfloat16, 3, "KEPT")])
def test_ragged_products_store_as_the_rule_says(route, M, N, K, out, shift, form):
    check_form(route, 0, route.BLOCK, M, N, K, out, shift, form)


# 2 MB of C whose rows start on lines, 4 and 16 MB of others, and an address inside a line; rings of three and six slots, the wide tile
@pytest.mark.parametrize("M,N,out,shift,form", [
    (255, 4096, torch.bfloat16, 0, "PIECES"), (256, 4096, torch.bfloat16, 0, "OUT"), (256, 4096, torch.bfloat16, 8, "PIECES"), (2100, 4096, torch.bfloat16, 0, "OUT"),
    (2100, 4096, torch.bfloat16, 8, "KEPT"), (511, 4104, torch.bfloat16, 0, "PIECES"), (512, 4104, torch.bfloat16, 0, "OUT"), (2044, 4104, torch.bfloat16, 0, "OUT"),
    (2045, 4104, torch.bfloat16, 0, "KEPT"), (127, 4096, torch.float32, 0, "PIECES"), (128, 4096, torch.float32, 0, "OUT"), (255, 4104, torch.float32, 0, "PIECES"),
    (256, 4104, torch.float32, 0, "OUT"), (1022, 4104, torch.float32, 0, "OUT"), (1023, 4104, torch.float32, 0, "KEPT"), (1100, 4096, torch.float32, 4, "KEPT")])
@pytest.mark.parametrize("kernel", [23, 24, 26])
def test_block_kernel_stores_as_the_rule_says(route, kernel, M, N, out, shift, form):
    check_form(route, kernel, kernel, M, N, 384, out, shift, form)


@pytest.mark.parametrize("M,N,out,shift,form", [
    (2044, 4104, torch.bfloat16, 0, "OUT"), (2045, 4104, torch.bfloat16, 0, "KEPT"), (2100, 4096, torch.bfloat16, 0, "OUT"), (2100, 4096, torch.bfloat16, 8, "KEPT"),
    (1022, 4104, torch.float32, 0, "OUT"), (1023, 4104, torch.float32, 0, "KEPT"), (1100, 4096, torch.float32, 4, "KEPT")])
@pytest.mark.parametrize("kernel", [5, 6, 17])
def test_tiled_kernel_stores_as_the_rule_says(route, kernel, M, N, out, shift, form):
    check_form(route, kernel, kernel, M, N, 384, out, shift, form)


def check_form(route, kernel, code, M, N, K, out, shift, form):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as hk

    tk, pad = hk.tk_kernel, 512
    g = torch.Generator(device="cuda").manual_seed(M + N)
    A, As = hk.quantize(torch.randn(M, K, device="cuda", generator=g), 2)
    B, Bs = hk.quantize(torch.randn(N, K, device="cuda", generator=g).mul_(0.05), 2)
    whole = torch.full((2 * pad + M * N,), 7.0, dtype=out, device="cuda")
    C = whole[pad + shift : pad + shift + M * N].view(M, N)
    taken = route.gemm(A, B, As, Bs, C, M, N, K, kernel=kernel, k_split=1)
    assert taken == code and route.memory == getattr(route, form), (taken, route.memory)
    assert (whole[: pad + shift] == 7).all() and (whole[pad + shift + M * N :] == 7).all()
    want = torch.empty(M, N, dtype=out, device="cuda")
    prev = tk.set_kernel(1)  # one wave per tile: the same sums
    try:
        tk.dispatch_micro(A, B, As, Bs, want, 2, 2)
    finally:
        tk.set_kernel(prev)
    assert torch.equal(C, want)
