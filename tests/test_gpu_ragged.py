"""Sizes and alignments that the aligned kernels do not take (N % 8, K % 128, pointers off 16 bytes), through the automatic
path: the block kernel's ragged instantiations against the CPU oracle, at the edges of their tiles and K-tiles.  Bound: every
product and partial sum of these inputs is exact in fp32 up to the sum's own rounding, so the fp32 result is held to 1e-5 of
the oracle's (its metric), the bf16 result to the rounding of that fp32 result, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import c_oracle as co
from oracle import mxfp6_oracle as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as m

    return m


def at(a, off):
    """`a` on the GPU at a pointer `off` bytes past 256-byte alignment, NaN bit patterns (0xff) around it."""
    raw = np.ascontiguousarray(a).view(np.uint8).reshape(-1)
    buf = torch.full((raw.size + 1024,), 255, dtype=torch.uint8, device="cuda")
    buf[256 + off:256 + off + raw.size] = torch.from_numpy(raw).cuda()
    return buf[256 + off:256 + off + raw.size].view(*a.shape)


def call(hk, A, B, As, Bs, M, N, fa, fb, dtype, off_c=0, shares=0, **kw):
    guard = torch.full((M * N + 64,), 7.0, dtype=dtype, device="cuda")
    C = guard[16 + off_c:16 + off_c + M * N].view(M, N)
    prev = hk.tk_kernel.set_k_split(shares)
    try:
        hk.dispatch_micro(A, B, As, Bs, C, fa, fb, **kw)
        torch.cuda.synchronize()
    finally:
        hk.tk_kernel.set_k_split(prev)
    assert bool((guard[:16 + off_c] == 7.0).all()) and bool((guard[16 + off_c + M * N:] == 7.0).all())
    return C


@pytest.mark.parametrize("M,N,K", [(1, 1, 160), (128, 128, 160), (129, 127, 288), (127, 129, 224), (5, 131, 2080), (257, 255, 1056), (130, 1001, 992),
                                   (64, 8, 4064), (33, 4, 8224), (300, 12, 640), (200, 260, 384), (1, 5003, 2880), (500, 515, 2880), (1000, 1001, 96)])
@pytest.mark.parametrize("fa,fb,shares", [(2, 2, 0), (2, 2, 1), (3, 2, 2), (2, 3, -1)])
def test_ragged_sizes_vs_oracle(hk, M, N, K, fa, fb, shares):
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(M + K)), fa)
    bp, bsc = co.quantise(o.make_source("weights_outliers", (N, K), np.random.default_rng(N + K)), fb)
    ref = o.gemm_ref(ap, bp, asc, bsc, fa, fb, acc=np.float64)
    ops = [at(x, 0) for x in (ap, bp, asc, bsc)]
    got = call(hk, *ops, M, N, fa, fb, torch.float32, shares=shares).cpu().numpy()
    assert np.isfinite(got).all() and o.rel_err(got, ref) <= 1e-5
    c16 = call(hk, *ops, M, N, fa, fb, torch.bfloat16, shares=shares)
    assert np.array_equal(c16.view(torch.int16).cpu().numpy().view(np.uint16), o.f32_to_bf16_bits(got))


@pytest.mark.parametrize("M,N,K,la", [(70, 136, 640, 0), (64, 136, 640, 1), (200, 96, 1056, 0)])
def test_ragged_alignment_and_fused_epilogue(hk, M, N, K, la):
    """Operands at every alignment the entry points take (4 bytes, scales and C any element), tile-major A, fused epilogue."""
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(1)), 2)
    bp, bsc = co.quantise(o.make_source("weights", (N, K), np.random.default_rng(2)), 2)
    ref = o.gemm_ref(ap, bp, asc, bsc, acc=np.float64)
    tiled = (o.tile_operand(ap), o.tile_scales(asc)) if la else (ap, asc)
    for oa, ob, osa, osb, oc in ((4, 0, 0, 0, 0), (0, 12, 0, 0, 1), (0, 0, 1, 2, 3), (8, 4, 3, 1, 5)):
        ops = [at(tiled[0], oa), at(bp, ob), at(tiled[1], osa), at(bsc, osb)]
        got = call(hk, *ops, M, N, 2, 2, torch.float32, off_c=oc, layout_a=la).cpu().numpy()
        assert o.rel_err(got, ref) <= 1e-5, (oa, ob, osa, osb, oc)
        bias = torch.randn(N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
        fused = call(hk, *ops, M, N, 2, 2, torch.float32, off_c=oc, layout_a=la, bias=bias, activation="relu").cpu().numpy()
        want = np.maximum(got + bias.cpu().numpy(), 0)  # one fp32 addition: exact to its rounding
        assert np.array_equal(fused, want.astype(np.float32)), (oa, ob, osa, osb, oc)


@pytest.mark.parametrize("N,first_is_odd_c", [(328, True), (344, False)])
def test_choice_is_per_alignment(hk, N, first_is_odd_c):
    """One shape twice: operands on 16 bytes with a C off 16 bytes (the decode kernel takes it), then scales one byte off with
    a C on 16 bytes (it does not), and in the other order: the first call's choice is not the second one's."""
    M, K = 16, 1536
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(4)), 2)
    bp, bsc = co.quantise(o.make_source("weights", (N, K), np.random.default_rng(5)), 2)
    ref = o.gemm_ref(ap, bp, asc, bsc, acc=np.float64)
    odd_c = ([at(x, 0) for x in (ap, bp, asc, bsc)], 1)
    odd_scales = ([at(ap, 0), at(bp, 0), at(asc, 1), at(bsc, 3)], 0)
    for ops, off_c in (odd_c, odd_scales) if first_is_odd_c else (odd_scales, odd_c):
        got = call(hk, *ops, M, N, 2, 2, torch.float32, off_c=off_c).cpu().numpy()
        assert o.rel_err(got, ref) <= 1e-5


@pytest.mark.parametrize("M,N,K,generic", [(200, 257, 288, True), (800, 511, 320, True), (100, 1003, 320, True), (200, 511, 480, True), (800, 257, 416, True),
                                           (64, 1003, 320, False), (16, 257, 288, False), (200, 3001, 288, False), (200, 101, 352, False), (200, 257, 512 + 32, False), (16, 5003, 288, False)])
def test_short_ragged_products_start_on_the_generic_kernel(hk, M, N, K, generic):
    """Both sides of the line between the one-wave-per-tile kernel and the block kernel, on the automatic path."""
    choice = hk.tk_kernel.kernel_choice(M, N, K)
    assert (choice == hk.tk_kernel.KERNEL_GENERIC) == generic and choice in (hk.tk_kernel.KERNEL_GENERIC, hk.tk_kernel.KERNEL_BLOCK)
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(M + K)), 2)
    bp, bsc = co.quantise(o.make_source("weights", (N, K), np.random.default_rng(N + K)), 2)
    got = call(hk, *(at(x, 0) for x in (ap, bp, asc, bsc)), M, N, 2, 2, torch.float32).cpu().numpy()
    assert o.rel_err(got, o.gemm_ref(ap, bp, asc, bsc, acc=np.float64)) <= 1e-5


@pytest.fixture
def padded():
    """Every ragged call of the measurement build on padded tile-major copies of its operands."""
    import ctypes

    from hipkittensp_amd import _lib

    P = _lib.probes()
    P.mxfp6_probe_padded.argtypes, P.mxfp6_probe_padded.restype = [ctypes.c_int], ctypes.c_int
    prev = P.mxfp6_probe_padded(1)
    yield P
    P.mxfp6_probe_padded(prev)


@pytest.mark.parametrize("M,N,K,offs,fa,fb", [(1, 1, 32, (0, 0, 0, 0, 0), 2, 2), (33, 65, 160, (4, 12, 1, 3, 1), 2, 3), (31, 264, 480, (8, 4, 2, 1, 0), 3, 2), (256, 256, 2080, (0, 0, 0, 0, 0), 2, 2),
                                              (129, 2048, 1056, (4, 8, 3, 2, 0), 2, 2), (100, 1003, 672, (0, 0, 0, 0, 3), 2, 2), (300, 40, 640, (4, 0, 0, 0, 0), 2, 2), (64, 8, 8224, (0, 0, 1, 1, 0), 2, 2)])
@pytest.mark.parametrize("f32", [0, 1])
def test_padded_copies_vs_oracle(hk, padded, M, N, K, offs, fa, fb, f32):
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(M + K)), fa)
    bp, bsc = co.quantise(o.make_source("weights_outliers", (N, K), np.random.default_rng(N + K)), fb)
    ref = o.gemm_ref(ap, bp, asc, bsc, fa, fb, acc=np.float64)
    ops = [at(x, off) for x, off in zip((ap, bp, asc, bsc), offs)]
    guard = torch.full((M * N + 64,), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
    C = guard[16 + offs[4]:16 + offs[4] + M * N]
    rc = padded.mxfp6_gemm_ex(*(t.data_ptr() for t in (*ops, C)), M, N, K, fa, fb, 0, 0, f32, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0 and bool((guard[:16 + offs[4]] == 7.0).all()) and bool((guard[16 + offs[4] + M * N:] == 7.0).all())
    got = C.view(M, N).float().cpu().numpy()
    # fp32: the sums' own bound; bf16: half a last place on top, 2^-8 of the value
    bound = 1e-5 * np.maximum(np.abs(ref), 0.01 * np.sqrt((ref**2).mean())) + (0 if f32 else np.abs(ref) * 2.0**-8)
    assert np.isfinite(got).all() and (np.abs(got - ref) <= bound).all()


@pytest.mark.parametrize("M,N,K,bf16", [(64, 96, 160, 1), (129, 1056, 672, 0), (200, 264, 2080, 1), (333, 515, 640, 1), (70, 8, 96, 0)])
def test_padded_linear_vs_oracle(hk, padded, M, N, K, bf16):
    """The quantiser writes the padded operand itself; NaN bit patterns in the workspace before the call reach nothing."""
    x = torch.from_numpy(o.make_source("normal", (M, K), np.random.default_rng(M)).astype(np.float32))
    x = x.to(torch.bfloat16) if bf16 else x
    ap, asc = co.quantise(x.float().numpy(), 2)
    bp, bsc = co.quantise(o.make_source("weights", (N, K), np.random.default_rng(N)), 2)
    ref = o.gemm_ref(ap, bp, asc, bsc, acc=np.float64)
    b, bs = at(bp, 0), at(bsc, 1)
    C = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for fill in (float("nan"), 0.0):
        big, junk = torch.full((2 * M, K + 128), fill, device="cuda"), torch.empty(2 * M, N, dtype=torch.bfloat16, device="cuda")
        prev = padded.mxfp6_probe_slice(-1)
        try:
            assert padded.mxfp6_linear(big.data_ptr(), 0, b.data_ptr(), bs.data_ptr(), junk.data_ptr(), M, N, K, 2, 2, 0, None, 0, 0, stream) == 0
            xc = at((x.view(torch.int16) if bf16 else x).numpy().view(np.uint8), 0)
            assert padded.mxfp6_linear(xc.data_ptr(), bf16, b.data_ptr(), bs.data_ptr(), C.data_ptr(), M, N, K, 2, 2, 0, None, 0, 0, stream) == 0
        finally:
            padded.mxfp6_probe_slice(prev)
        torch.cuda.synchronize()
        got = C.float().cpu().numpy()
        bound = 1e-5 * np.maximum(np.abs(ref), 0.01 * np.sqrt((ref**2).mean())) + np.abs(ref) * 2.0**-8
        assert np.isfinite(got).all() and (np.abs(got - ref) <= bound).all()


@pytest.mark.parametrize("M,N,K,pays", [(2604, 704, 5664, False), (2048, 3784, 3680, True), (4096, 1504, 3680, True), (2100, 5000, 4000, True)])
def test_padded_route_and_capture(hk, route, M, N, K, pays):
    """Products the choice gives to padded copies (and one that it does not): the bits of the block kernel's ragged instantiations (sums in the same order), and
    under capture on a stream without a workspace, where those run."""
    g = torch.Generator(device="cuda").manual_seed(M)
    (a, asc), (b, bsc) = hk.quantize(torch.randn(M, K, device="cuda", generator=g)), hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.02)
    prev, want, got = hk.tk_kernel.set_relayout(0), torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    try:
        hk.dispatch_micro(a, b, asc, bsc, want)
    finally:
        hk.tk_kernel.set_relayout(prev)
    copies = route.COPY_A | route.COPY_B
    assert route.gemm(a, b, asc, bsc, got, M, N, K) & copies == (copies if pays else 0)
    hk.dispatch_micro(a, b, asc, bsc, got)
    assert torch.equal(got, want)
    graph, C = torch.cuda.CUDAGraph(), torch.zeros(M, N, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        hk.dispatch_micro(a, b, asc, bsc, C)
    for _ in range(3):
        C.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want)


# kernel 2 is forced (unsplit: a K split takes no copies) where the choice would be another; MXFP6 output takes copies unforced only
@pytest.mark.parametrize("M,N,K,kernel", [(1001, 2056, 8192, 2), (31, 4104, 8192, 2), (2049, 1000, 16384, 2), (1793, 14336, 8192, 0), (4999, 2048, 16384, 0), (777, 6152, 16384, 2)])
@pytest.mark.parametrize("tile_b", [0, 1])
def test_relayout_of_rows_that_fill_no_row_tile(hk, route, M, N, K, kernel, tile_b):
    """The tiled kernel's pre-pass on operands whose rows end inside a row-tile: the bits of the row-major path, whose sums are in the
    same order, for every output type, with NaN patterns around the operands and in the workspace before the call."""
    if tile_b and N % 32:
        N -= N % 32
    g = torch.Generator(device="cuda").manual_seed(M)
    qa, qb = hk.quantize(torch.randn(M, K, device="cuda", generator=g)), hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.02, 2, tile_b)
    (a, asc), (b, bsc) = [[at(x.cpu().numpy(), 0).view(x.shape) for x in q] for q in (qa, qb)]
    T = hk.tk_kernel
    # which operands are copied: the one with fewer rows, and where that pays twice the other one
    copied = {(1001, 0): 1, (31, 0): 1, (2049, 0): 3, (1793, 0): 1, (4999, 0): 2, (777, 0): 1}.get((M, tile_b))
    prev_k, prev_split = T.set_kernel(kernel), T.set_k_split(1)
    try:
        for dtype in (torch.float32, torch.bfloat16, torch.uint8):
            outs = []
            for on in (0, 1, 1):
                if on and not outs[1:]:  # the stream's workspace full of NaN patterns
                    full = [torch.full((M, K // 4 * 3), 255, dtype=torch.uint8, device="cuda"), torch.full((M, K // 32), 255, dtype=torch.uint8, device="cuda")]
                    hk.dispatch_micro(*full[:1], b, *full[1:], bsc, torch.empty(M, N, device="cuda"), layout_b=tile_b)
                prev = T.set_relayout(on)
                try:
                    if dtype == torch.uint8 and N % 32 == 0:
                        C, S = torch.zeros(M, N // 4 * 3, dtype=dtype, device="cuda"), torch.zeros(M, N // 32, dtype=dtype, device="cuda")
                        if on and copied and not kernel:
                            assert route.gemm(a, b, asc, bsc, C, M, N, K, lb=tile_b, C_scale=S, k_split=1) == route.TILED | copied << 8
                        hk.dispatch_micro(a, b, asc, bsc, C, layout_b=tile_b, C_scale=S)
                        outs.append(torch.cat([C, S], 1))
                    elif dtype != torch.uint8:
                        C = torch.empty(M, N, dtype=dtype, device="cuda")
                        if on:
                            taken = route.gemm(a, b, asc, bsc, C, M, N, K, lb=tile_b, kernel=kernel, k_split=1)
                            assert taken & 0xff == route.TILED and (taken >> 8 == copied if copied else not taken & route.COPY_B)
                        hk.dispatch_micro(a, b, asc, bsc, C, layout_b=tile_b)
                        outs.append(C)
                finally:
                    T.set_relayout(prev)
            assert all(torch.equal(x, outs[0]) for x in outs[1:])
    finally:
        T.set_kernel(prev_k), T.set_k_split(prev_split)
