"""The linear layer's single native call (mxfp6_linear) against the two public calls it stands for, quantise then GEMM: the same
packed activations and the same kernels' sums, so the same bits wherever those are exact (these inputs' sums are), at the
edges of its layouts: below and above 64 rows, row counts that are no multiple of the 16 and 32 rows of a tile-major
chunk, K-tiles that fill no group of four."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as m

    return m


def steps(hk, layer, x):
    tk = hk.tk_kernel
    rows = x.numel() // x.shape[-1]
    xp, xs = tk.quantize(x.reshape(rows, -1), layer.fmt_x)
    C = torch.empty(rows, layer.out_features, dtype=torch.bfloat16, device="cuda")
    tk.dispatch_micro(xp, layer.weight_packed, xs, layer.weight_scale, C, layer.fmt_x, layer.fmt_w, 0, layer.layout_w, bias=layer.bias, activation=layer.activation)
    return C.view(*x.shape[:-1], -1)


@pytest.mark.parametrize("M", [1, 17, 63, 64, 65, 79, 80, 81, 97, 200, 257, 700])
@pytest.mark.parametrize("N,K", [(256, 512), (96, 640), (1000, 1152), (160, 96), (33, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_linear_is_quantise_then_gemm(hk, M, N, K, dtype):
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    layer = MXFP6Linear(torch.randn(N, K, device="cuda", generator=g) * 0.02, bias=torch.randn(N, device="cuda", generator=g).to(torch.bfloat16), activation="relu")
    for x in (torch.randn(M, K, device="cuda", generator=g).to(dtype), torch.randn(2, M, K, device="cuda", generator=g).to(dtype)):
        y = layer(x)
        assert y.shape == (*x.shape[:-1], N) and y.dtype == torch.bfloat16
        assert torch.equal(y, steps(hk, layer, x)), (M, N, K, x.shape)


def test_linear_streams_graphs_and_general_cases(hk):
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(5)
    layer = MXFP6Linear(torch.randn(512, 1024, device="cuda", generator=g) * 0.02)
    xs = [torch.randn(96, 1024, device="cuda", generator=g) for _ in range(2)]
    want = [steps(hk, layer, x) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]   # a workspace per stream
    out = [[], []]
    for _ in range(8):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                out[i].append(layer(xs[i]))
    torch.cuda.synchronize()
    assert all(torch.equal(y, want[i]) for i in range(2) for y in out[i])
    assert torch.equal(layer(xs[0].t().contiguous().t()), want[0])      # a view that is not contiguous
    assert torch.equal(layer(xs[0].to(torch.float16).to(torch.float32)), steps(hk, layer, xs[0].to(torch.float16).float()))
    # captured on a stream with a workspace and on one without; replayed with other work in between
    x = xs[0].clone()
    for s in (streams[0], torch.cuda.Stream()):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            y = layer(x)
        for i in (1, 0, 1):
            x.copy_(xs[i])
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want[i])
            layer(xs[0])
            torch.cuda.synchronize()
    with pytest.raises(RuntimeError):
        layer(torch.randn(4, 1000, device="cuda"))   # K of another layer


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,K", [(32, 128), (64, 640), (32, 896), (96, 1152)])
def test_tile_major_scales_are_padded_with_zeros(hk, rows, K, dtype):
    from hipkittensp_amd import _lib

    x = torch.randn(rows, K, device="cuda", generator=torch.Generator(device="cuda").manual_seed(K)).to(dtype)
    w = (K + 511) // 512 * 16
    p = torch.empty(rows, K // 4 * 3, dtype=torch.uint8, device="cuda")
    s = torch.full((rows, w), 255, dtype=torch.uint8, device="cuda")
    fn = _lib.lib().mxfp6_quantize_bf16 if dtype == torch.bfloat16 else _lib.lib().mxfp6_quantize_ex
    assert fn(x.data_ptr(), p.data_ptr(), s.data_ptr(), rows, K, 2, 1, torch.cuda.current_stream().cuda_stream) == 0
    pr, sr = hk.quantize(x, 2)
    assert torch.equal(s, hk.tile_scales(sr, K)) and torch.equal(p, hk.tile_operand(pr))


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("N,K", [(40, 512), (4096, 4096), (1000, 1536), (512, 16384), (5000, 1024), (8200, 1024), (16384, 512), (33000, 512)])
@pytest.mark.parametrize("fmt_x,fmt_w", [(2, 2), (3, 2), (2, 3)])
def test_few_rows_quantised_inside_the_gemm(hk, M, N, K, fmt_x, fmt_w):
    """bf16 activations of up to four rows, which the decode kernel quantises itself: the bits of quantise, then GEMM, for every
    workgroup shape it has (few and many rows of weights, K split between workgroups), for blocks of zeros, for subnormal
    and very large values and for NaN (each block's own)."""
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    layer = MXFP6Linear(torch.randn(N, K, device="cuda", generator=g) * 0.02, fmt_w=fmt_w, fmt_x=fmt_x, bias=torch.randn(N, device="cuda", generator=g), activation="silu")
    guard = torch.randn(M * K + 4096, device="cuda", generator=g).to(torch.bfloat16)
    guard[M * K:] = float("nan")
    x = guard[:M * K].view(M, K)
    assert torch.equal(layer(x), steps(hk, layer, x))
    x[0, 32:64] = 0
    x[M - 1, 64:96] *= 1e-39
    x[M - 1, K - 32:] *= 1e30
    y, want = layer(x), steps(hk, layer, x)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    x[0, 5] = float("nan")
    y, want = layer(x), steps(hk, layer, x)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("kernel,shares,M,N,K,tile_b", [(23, 1, 129, 4096, 640, True), (24, 1, 500, 1056, 2176, False), (26, 1, 300, 2080, 640, True), (26, 1, 128, 96, 128, False),
                                                        (22, 3, 257, 2048, 4096, False), (22, 5, 90, 1056, 2816, True), (0, 0, 256, 8192, 28672, True),
                                                        (0, 0, 300, 12064, 4096, False), (0, 0, 384, 4096, 640, True), (0, 0, 700, 8896, 640, False), (0, 0, 1500, 11008, 4096, True), (0, 0, 4096, 2048, 512, True)])
@pytest.mark.parametrize("fmt_c", [2, 3])
def test_fp6_output_of_the_block_kernel_and_the_k_splits(hk, kernel, shares, M, N, K, tile_b, fmt_c):
    """Bit for bit the quantiser applied to the fp32 result of the same call, which the same kernel computes: edge tiles, an
    odd number of 32-column tiles, several shares; blocks of zeros, of NaN and of infinities; outputs that start 8 bytes past a
    multiple of 16; nothing written around them."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, asc = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
    lb = hk.LAYOUT_TILE if tile_b else hk.LAYOUT_ROW
    b, bsc = hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.05, 2, lb)
    bias = torch.randn(N, device="cuda", generator=g)
    cs = torch.rand(N, device="cuda", generator=g) + 0.5
    rs = torch.rand(M, device="cuda", generator=g) + 0.5
    cs[:32], rs[M - 1] = 0.0, float("nan")
    cs[64:65] = float("inf")
    prev, prev_split = hk.tk_kernel.set_kernel(kernel), hk.tk_kernel.set_k_split(shares)
    try:
        for kw in (dict(), dict(bias=bias, row_scale=rs, activation="gelu"), dict(col_scale=cs, row_scale=rs, activation="relu")):
            C = torch.empty(M, N, dtype=torch.float32, device="cuda")
            hk.dispatch_micro(a, b, asc, bsc, C, 2, 2, hk.LAYOUT_ROW, lb, **kw)
            want, want_s = hk.quantize(C, fmt_c)
            n, m = M * (N // 4 * 3), M * (N // 32)
            raw, raw_s = torch.full((n + 64,), 0xAA, dtype=torch.uint8, device="cuda"), torch.full((m + 64,), 0xAA, dtype=torch.uint8, device="cuda")
            P, S = raw[8:8 + n].view(M, -1), raw_s[8:8 + m].view(M, -1)
            hk.dispatch_micro(a, b, asc, bsc, P, 2, 2, hk.LAYOUT_ROW, lb, C_scale=S, fmt_c=fmt_c, **kw)
            assert torch.equal(S, want_s) and torch.equal(P, want)
            for r, k in ((raw, n), (raw_s, m)):
                assert (r[:8] == 0xAA).all() and (r[8 + k:] == 0xAA).all()
    finally:
        hk.tk_kernel.set_kernel(prev)
        hk.tk_kernel.set_k_split(prev_split)


@pytest.mark.parametrize("M", [65, 97, 257, 300])
@pytest.mark.parametrize("N,K", [(256, 512), (96, 640)])
def test_linear_on_the_four_wave_kernel(hk, M, N, K):
    """Row counts that end in a partial row-tile of the packed activations: the last tile's rows are multiplied whole."""
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    layer = MXFP6Linear(torch.randn(N, K, device="cuda", generator=g) * 0.02)
    x = torch.randn(M, K, device="cuda", generator=g)
    want = steps(hk, layer, x)
    prev = hk.tk_kernel.set_kernel(hk.tk_kernel.KERNEL_TILED_4WAVE)
    try:
        assert torch.equal(layer(x), want)
    finally:
        hk.tk_kernel.set_kernel(prev)


@pytest.mark.parametrize("M", [65, 97, 127])
@pytest.mark.parametrize("kernel", [3, 4, 7, 16, 21])
def test_linear_on_forced_kernels_of_row_major_activations(hk, M, kernel):
    """Kernels that take a row-major A only run the layer at row counts that fill no row-tile.  (Sums of 1024 products of
    4-bit significands are exact in any order.)"""
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(M)
    layer = MXFP6Linear(torch.randn(256, 1024, device="cuda", generator=g) * 0.02, activation="relu")
    x = torch.randn(M, 1024, device="cuda", generator=g)
    want = steps(hk, layer, x)
    prev = hk.tk_kernel.set_kernel(kernel)
    try:
        assert torch.equal(layer(x), want)
    finally:
        hk.tk_kernel.set_kernel(prev)


def test_graphs_of_one_stream_share_no_activations(hk):
    """Two graphs of a layer captured on one stream that has run it before, replayed side by side on two others, beside the layer
    itself on the capture stream: the packed activations of each are its own."""
    from hipkittensp_amd import _lib
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(8)
    M, N, K = 200, 512, 8192
    layer = MXFP6Linear(torch.randn(N, K, device="cuda", generator=g) * 0.02)
    xs = [torch.randn(M, K, device="cuda", generator=g) for _ in range(3)]
    want = [steps(hk, layer, x) for x in xs]
    capture, streams = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    prev = hk.tk_kernel.set_k_split(1)   # a K split's partial sums are the stream's, as the header says
    try:
        with torch.cuda.stream(capture):
            layer(xs[2])
        torch.cuda.synchronize()
        graphs, ys = [], []
        for i in range(2):
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=capture):
                if i == 0:
                    C = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
                    assert _lib.lib().mxfp6_linear(xs[0].data_ptr(), 0, layer.weight_packed.data_ptr(), layer.weight_scale.data_ptr(), C.data_ptr(), M, N, K,
                                                   2, 2, layer.layout_w, None, 0, 0, torch.cuda.current_stream().cuda_stream) == -11   # MXFP6_EWORKSPACE
                ys.append(layer(xs[i]))
            graphs.append(graph)
        for _ in range(20):
            for s, graph in zip(streams, graphs):
                with torch.cuda.stream(s):
                    graph.replay()
            with torch.cuda.stream(capture):
                y = layer(xs[2])
            torch.cuda.synchronize()
            for got, w in zip((*ys, y), want):
                assert torch.equal(got, w)
    finally:
        hk.tk_kernel.set_k_split(prev)


@pytest.mark.parametrize("M", [1, 4])
def test_decode_rows_are_captured_in_one_launch(hk, M):
    """Up to four bf16 rows need no workspace for their activations: mxfp6_linear itself is captured, on a stream that has none."""
    from hipkittensp_amd import _lib
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(9)
    layer = MXFP6Linear(torch.randn(512, 1024, device="cuda", generator=g) * 0.02)
    x = torch.randn(M, 1024, device="cuda", generator=g).to(torch.bfloat16)
    C, graph = torch.zeros(M, 512, dtype=torch.bfloat16, device="cuda"), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        assert _lib.lib().mxfp6_linear(x.data_ptr(), 1, layer.weight_packed.data_ptr(), layer.weight_scale.data_ptr(), C.data_ptr(), M, 512, 1024,
                                       2, 2, layer.layout_w, None, 0, 0, torch.cuda.current_stream().cuda_stream) == 0
    for _ in range(3):
        x.copy_(torch.randn(M, 1024, device="cuda", generator=g))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, steps(hk, layer, x))


@pytest.mark.parametrize("M,N,K,act", [(512, 11008, 8192, "gelu"), (1024, 5120, 8192, "none"), (256, 8192, 28672, "relu"), (64, 8192, 28672, "none")])
def test_fp6_output_is_captured_on_a_stream_without_workspace(hk, M, N, K, act):
    """A K split needs its workspace and the decode kernels the fp32 one; a capture on a stream that has neither records a kernel
    that needs none.  Its fp32 sums may differ from the eager call's in their last place (2^-24), which moves a code only next
    to a rounding boundary of its 2^-4 steps: at most one byte in 10 000 differs."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a, asc = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
    b, bsc = hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.02, 2, hk.LAYOUT_TILE)
    mk = lambda: (torch.zeros(M, N // 4 * 3, dtype=torch.uint8, device="cuda"), torch.zeros(M, N // 32, dtype=torch.uint8, device="cuda"))
    want, got = mk(), mk()
    call = lambda out: hk.dispatch_micro(a, b, asc, bsc, out[0], 2, 2, hk.LAYOUT_ROW, hk.LAYOUT_TILE, C_scale=out[1], activation=act)
    call(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        call(got)
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all((x != y).float().mean().item() <= 1e-4 for x, y in zip(got, want))
        call(want)


def test_exceptions_in_the_binding_are_python_errors(hk):
    """Tensors whose sizes or memory cannot be read (nested ones, those a fake-tensor mode makes) end in a Python error, and the
    calls after them work."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(8, 512, device="cuda", generator=g)
    layer = MXFP6Linear(torch.randn(64, 512, device="cuda", generator=g) * 0.02)
    want, (p, s) = steps(hk, layer, x), hk.quantize(x)
    nested = torch.nested.nested_tensor([torch.zeros(24, dtype=torch.uint8), torch.zeros(48, dtype=torch.uint8)]).cuda()
    C = torch.empty(8, 64, dtype=torch.bfloat16, device="cuda")
    for args in ((nested, p, s, s, C), (p, nested, s, s, C), (p, p, nested, s, C), (p, p, s, s, nested)):
        with pytest.raises(RuntimeError):
            hk.dispatch_micro(*args)
    with pytest.raises(RuntimeError):
        hk.quantize(torch.nested.nested_tensor([torch.zeros(32), torch.zeros(64)]).cuda())
    with FakeTensorMode(allow_non_fake_inputs=True), pytest.raises(RuntimeError):
        hk.quantize(x)
    assert torch.equal(layer(x), want) and torch.equal(hk.quantize(x)[0], p)


@pytest.mark.parametrize("M,N,K,act", [(8192, 8192, 256, "gelu"), (4096, 16384, 384, "silu"), (8192, 9216, 128, "gelu")])
def test_activations_on_outputs_past_the_last_level_cache(hk, M, N, K, act):
    """From 256 MB of fp32 output on the choice counts an activation for bf16 and MXFP6 output only: other tiles, the same sums, so
    the bf16 result is the rounded fp32 one and the MXFP6 one its quantisation, bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a, asc = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
    b, bsc = hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.1, 2, hk.LAYOUT_TILE)
    bias = torch.randn(N, device="cuda", generator=g)
    C = torch.empty(M, N, dtype=torch.float32, device="cuda")
    C16 = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    P, S = torch.empty(M, N // 4 * 3, dtype=torch.uint8, device="cuda"), torch.empty(M, N // 32, dtype=torch.uint8, device="cuda")
    for out, kw in ((C, {}), (C16, {}), (P, dict(C_scale=S))):
        hk.dispatch_micro(a, b, asc, bsc, out, 2, 2, hk.LAYOUT_ROW, hk.LAYOUT_TILE, bias=bias, activation=act, **kw)
    want, want_s = hk.quantize(C)
    assert torch.equal(C16, C.to(torch.bfloat16)) and torch.equal(P, want) and torch.equal(S, want_s)


def test_activation_is_read_per_call(hk):
    """A layer's activation may be set after it was made (or come from a module saved without any other state of it); what is no name
    of one is refused."""
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(6)
    layer = MXFP6Linear(torch.randn(64, 512, device="cuda", generator=g) * 0.02)
    for M in (3, 8):
        x = torch.randn(M, 512, device="cuda", generator=g).to(torch.bfloat16)
        for act in ("none", "relu", "gelu", "silu"):
            layer.activation = act
            assert torch.equal(layer(x), steps(hk, layer, x))
        for act in (None, 1, "tanh"):
            layer.activation = act
            with pytest.raises((RuntimeError, TypeError, KeyError, ValueError)):
                layer(x)


def us_per_call(call, n=200):
    """Best of five runs"""
    times = []
    for _ in range(5):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        for i in range(20 + n):
            if i == 20:
                start.record()
            call()
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end) * 1000 / n)
    return min(times)


def test_a_call_that_asks_twice_for_its_kernel_remembers_both_answers(hk):
    """MXFP6 output of a few rows goes through fp32 sums and the quantiser, and a kernel is chosen twice in the call.  Both choices are
    remembered: the call takes no longer than the two public calls it stands for (8.5 us).  Two choices worked out anew
    every time made it 20 us."""
    g = torch.Generator(device="cuda").manual_seed(2)
    M, N, K = 6, 4992, 2560
    a, asc = hk.quantize(torch.randn(M, K, device="cuda", generator=g))
    b, bsc = hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.02, 2, hk.LAYOUT_TILE)
    C = torch.empty(M, N, dtype=torch.float32, device="cuda")
    P, S = torch.empty(M, N // 4 * 3, dtype=torch.uint8, device="cuda"), torch.empty(M, N // 32, dtype=torch.uint8, device="cuda")
    ops = (a, b, asc, bsc)
    one = us_per_call(lambda: hk.dispatch_micro(*ops, P, 2, 2, hk.LAYOUT_ROW, hk.LAYOUT_TILE, C_scale=S, activation="relu"))
    two = us_per_call(lambda: (hk.dispatch_micro(*ops, C, 2, 2, hk.LAYOUT_ROW, hk.LAYOUT_TILE, activation="relu"), hk.quantize(C)))
    assert one <= 1.2 * two + 0.5


def test_a_layer_that_asks_twice_for_its_kernel_remembers_both_answers(hk):
    """Up to four bf16 rows a layer first asks whether the decode kernel, which would quantise them itself, is the choice, then, as here
    where it is not, for the GEMM with its activation: no longer than the two public calls either."""
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(2)
    layer = MXFP6Linear(torch.randn(12288, 512, device="cuda", generator=g) * 0.02, activation="relu")
    x = torch.randn(4, 512, device="cuda", generator=g).to(torch.bfloat16)
    one, two = us_per_call(lambda: layer(x)), us_per_call(lambda: steps(hk, layer, x))
    assert one <= 1.2 * two + 0.5


@pytest.mark.parametrize("rows,dtype,bound", [(6144, torch.float32, 2.0), (8192, torch.bfloat16, 1.97)])
def test_quantiser_reads_an_input_that_is_in_the_cache_from_there(hk, rows, dtype, bound):
    """An input below the size of the last-level cache, quantised again and again, against one of half its rows: 35.1 us against 18.9 for 192
    MB of fp32 and 28.9 against 15.5 for 128 MB of bf16 (a ratio of 1.86 each), 40.4 and 31.9 (2.14 and 2.06) when it is read past that cache."""
    x = torch.randn(rows, 8192, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).to(dtype)
    half = x[:rows // 2].contiguous()
    ratios = []
    for _ in range(3):
        ratios.append(us_per_call(lambda: hk.quantize(x, 2, hk.LAYOUT_TILE), 60) / us_per_call(lambda: hk.quantize(half, 2, hk.LAYOUT_TILE), 60))
        if ratios[-1] <= bound:
            break
    assert min(ratios) <= bound, ratios
