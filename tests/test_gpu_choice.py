"""The kernel choice between K splits and their neighbours, timed as a program's calls: new activations and another layer's weights every
time."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as m

    return m


def ratios_to_the_best_forced_kernel(hk, M, N, K, la, lb, bound):
    """Up to three measurements, until one is within the bound."""
    tk = hk.tk_kernel
    g = torch.Generator(device="cuda").manual_seed(M + N)
    acts = [hk.quantize(torch.randn(M, K, device="cuda", generator=g), 2, la) for _ in range(3)]
    b = hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.02, 2, lb)
    weights = [b] + [(b[0].clone(), b[1].clone()) for _ in range(min(15, 400_000_000 // b[0].numel()))]
    outs = [torch.empty(M, N, dtype=torch.bfloat16, device="cuda") for _ in range(3)]

    def us(kernel, k_split):
        prev = tk.set_kernel(kernel), tk.set_k_split(k_split)
        try:
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            for i in range(110):
                if i == 10:
                    start.record()
                (a, asc), (w, ws) = acts[i % 3], weights[i % len(weights)]
                tk.dispatch_micro(a, w, asc, ws, outs[i % 3], 2, 2, la, lb)
            end.record()
            end.synchronize()
        finally:
            tk.set_kernel(prev[0]), tk.set_k_split(prev[1])
        return start.elapsed_time(end) * 10

    forced = [(k, s) for k in (tk.KERNEL_TILED_256, tk.KERNEL_TILED_128, tk.KERNEL_BLOCK) for s in (1, -1)] + [(tk.KERNEL_BLOCK_WIDE, 0)]
    if M <= 128:
        forced += [(tk.KERNEL_SKINNY, 0), (tk.KERNEL_RING, 0)]
    ratios = []
    for _ in range(3):
        ratios.append(us(tk.KERNEL_AUTO, 0) / min(us(*f) for f in forced))
        if ratios[-1] <= bound:
            break
    return ratios


@pytest.mark.parametrize("M,N,K,la,lb", [(256, 8192, 28672, 0, 1), (320, 4096, 24576, 0, 1), (192, 7168, 20480, 0, 1), (768, 3072, 12288, 1, 0), (2048, 4096, 8192, 1, 0)])
def test_choice_with_new_activations_per_call(hk, M, N, K, la, lb):
    """Within 4 % of the best forced kernel (runs of one form differ by up to 2 %; a calibration with one set of activations for
    all its launches chose a kernel 5 to 10 % behind at the second shape and 3 % at the first)."""
    ratios = ratios_to_the_best_forced_kernel(hk, M, N, K, la, lb, 1.04)
    assert min(ratios) <= 1.04, ratios


@pytest.mark.parametrize("M,N,K,la,lb", [(28, 9216, 9216, 0, 1), (2304, 9216, 9216, 0, 0), (1280, 3328, 16640, 0, 1), (104, 45056, 3584, 0, 0)])
def test_choice_at_widths_of_the_second_calibration_set(hk, M, N, K, la, lb):
    """Within 8 %; from the first set alone the choice was 14 to 34 % behind here."""
    ratios = ratios_to_the_best_forced_kernel(hk, M, N, K, la, lb, 1.08)
    assert min(ratios) <= 1.08, ratios


@pytest.mark.parametrize("M,N,K,la,lb", [(28, 2688, 10752, 0, 1), (32, 3072, 7168, 0, 1), (25, 4224, 11776, 0, 1), (64, 2944, 13824, 0, 1)])
def test_choice_of_small_products_with_weights_from_memory(hk, M, N, K, la, lb):
    """Within 8 %; the slice kernel, whose model knew weights from the cache only, was chosen here and 14 to 36 % behind."""
    ratios = ratios_to_the_best_forced_kernel(hk, M, N, K, la, lb, 1.08)
    assert min(ratios) <= 1.08, ratios


@pytest.mark.parametrize("M,N,K,lb", [(2, 7552, 8320, 1), (35, 3584, 10624, 1), (11, 11392, 4352, 1), (46, 10880, 2688, 0)])
def test_slice_kernel_with_weights_from_memory(hk, route, M, N, K, lb):
    """Its modelled time from memory lies up to 5 % below the block kernel's, and it is 13 to 25 % faster: a margin there kept it out."""
    g = torch.Generator(device="cuda").manual_seed(M)
    a, asc = hk.quantize(torch.randn(M, K, device="cuda", generator=g), 2)
    b, bsc = hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.02, 2, lb)
    C = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    assert route.gemm(a, b, asc, bsc, C, M, N, K, lb=lb) & 0xFF == route.SLICE
