"""MXFP6 output of the decode kernels: every workgroup shape of the skinny kernel and the ring kernel, unsplit and with a K split,
write bit for bit the quantiser's result on the same call's fp32 output (the sums and their order are the same)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as m

    return m


# kernel 0: the library's choice; 3 - 21: the skinny kernel (8: 16 rows of B a workgroup, which goes through a workspace); 28: ring
@pytest.mark.parametrize("kernel,M,N,K", [
    (0, 1, 8192, 4096), (0, 23, 14336, 4096), (0, 64, 9216, 8192), (0, 128, 8192, 28672), (0, 7, 2048, 8192), (0, 16, 28672, 512),
    (3, 33, 96, 1024), (7, 1, 32, 512), (7, 31, 4128, 2560), (7, 65, 64, 1536), (7, 128, 160, 512), (8, 5, 64, 1024), (9, 16, 96, 2560),
    (9, 17, 96, 512), (9, 64, 32, 1024), (9, 127, 96, 1024), (10, 3, 64, 12288), (12, 32, 224, 16384), (16, 9, 160, 1024),
    (19, 20, 96, 3072), (20, 50, 160, 8192), (21, 100, 96, 16384),
    (28, 1, 32, 512), (28, 32, 128, 2560), (28, 33, 160, 8192), (28, 64, 288, 1024), (28, 65, 96, 16384), (28, 200, 416, 4096)])
def test_decode_kernels_store_mxfp6(hk, kernel, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    fa, fb, tile = ((2, 2, 0), (3, 2, 1), (2, 3, 1))[(M + N // 32) % 3]
    a, asc = hk.quantize(torch.randn(M, K, device="cuda", generator=g), fa)
    b, bsc = hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.05, fb, tile)
    bias = torch.randn(N, device="cuda", generator=g)
    bias[1], bias[N - 2], bias[N - 1] = float("nan"), float("inf"), 1e-42
    rs = torch.rand(M, device="cuda", generator=g) + 0.5
    prev = hk.tk_kernel.set_kernel(kernel)
    try:
        for fmt_c, kw in ((2, {}), (3, dict(bias=bias, row_scale=rs, activation="silu"))):
            C = torch.empty(M, N, dtype=torch.float32, device="cuda")
            hk.dispatch_micro(a, b, asc, bsc, C, fa, fb, 0, tile, **kw)
            P, S = (torch.full((M * w + 128,), 0xAA, dtype=torch.uint8, device="cuda") for w in (N // 4 * 3, N // 32))
            p, s = P[64:64 + M * (N // 4 * 3)].view(M, -1), S[64:64 + M * (N // 32)].view(M, -1)
            for _ in range(2):  # a K split's counters are back at zero
                hk.dispatch_micro(a, b, asc, bsc, p, fa, fb, 0, tile, C_scale=s, fmt_c=fmt_c, **kw)
            want_p, want_s = hk.quantize(C, fmt_c)
            assert torch.equal(p, want_p) and torch.equal(s, want_s)
            for t in (P, S):
                assert bool((t[:64] == 0xAA).all()) and bool((t[-64:] == 0xAA).all())
    finally:
        hk.tk_kernel.set_kernel(prev)


@pytest.mark.parametrize("M,N,K,off", [(793, 1024, 640, (4, 0)), (400, 1536, 1024, (0, 1)), (130, 2560, 512, (8, 2)), (96, 768, 6144, (4, 0))])
def test_mxfp6_output_beside_fp32_output_off_16_bytes(hk, M, N, K, off):
    """A (its packed bytes, its scales) off 16 bytes against prepared weights: MXFP6 output has the bits of the quantised fp32 output here
    too, on sums that show their order (every other K-block of the first half is 2^18 times the rest and cancels)."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = ((torch.randn(r, K, device="cuda", generator=g) * c).view(r, K // 32, 32) for r, c in ((M, 1.0), (N, 0.02)))
    q = K // 128
    x[:, :q:2] *= 2.0**18
    x[:, q:2 * q:2], w[:, q:2 * q:2] = -x[:, :q:2], w[:, :q:2]
    b, bsc = hk.quantize(w.reshape(N, K), 2, 1)

    def moved(t, by):
        buf = torch.empty(t.numel() + 256, dtype=torch.uint8, device="cuda")
        out = buf[by:by + t.numel()].view(t.shape)
        return out.copy_(t)

    a, asc = (moved(t, by) for t, by in zip(hk.quantize(x.reshape(M, K), 2), off))
    C = torch.empty(M, N, device="cuda")
    p, s = torch.empty(M, N // 4 * 3, dtype=torch.uint8, device="cuda"), torch.empty(M, N // 32, dtype=torch.uint8, device="cuda")
    hk.dispatch_micro(a, b, asc, bsc, C, layout_b=1)
    hk.dispatch_micro(a, b, asc, bsc, p, layout_b=1, C_scale=s)
    want_p, want_s = hk.quantize(C, 2)
    assert torch.equal(p, want_p) and torch.equal(s, want_s)


def test_decode_output_under_capture_without_a_workspace(hk):
    M, N, K = 24, 8192, 4096
    g = torch.Generator(device="cuda").manual_seed(3)
    a, asc = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
    b, bsc = hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.05)
    C = torch.empty(M, N, dtype=torch.float32, device="cuda")
    p, s = torch.zeros(M, N // 4 * 3, dtype=torch.uint8, device="cuda"), torch.zeros(M, N // 32, dtype=torch.uint8, device="cuda")
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        hk.dispatch_micro(a, b, asc, bsc, p, C_scale=s)
        hk.dispatch_micro(a, b, asc, bsc, C)
    for _ in range(3):
        a2, as2 = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
        a.copy_(a2), asc.copy_(as2)
        p.zero_(), s.zero_(), C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        # no workspace, so no K split between workgroups: kernels may differ between the outputs, by the order of their sums
        dq_p, dq_s = hk.quantize(C)
        assert (p != dq_p).float().mean() < 1e-3 and torch.equal(s, dq_s)
