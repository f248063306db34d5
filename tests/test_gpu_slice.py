"""The slice kernel (tiles of 32 or 64 rows and columns, K dealt to waves and workgroups): every tile shape at the edges of its
tiles and chunks against the CPU oracle, and the routes that lead to it.  Bound as for the other kernels: products and partial
sums of these inputs are exact in fp32 up to the sum's own rounding, 1e-5 in the oracle's metric."""
import ctypes

import numpy as np
import pytest
import torch

from hipkittensp_amd import _lib
from oracle import c_oracle as co
from oracle import mxfp6_oracle as o

pytestmark = pytest.mark.gpu

PLANS = [(1, 1, 4), (1, 1, 8), (1, 2, 4), (1, 2, 8), (2, 2, 6)]


@pytest.fixture(scope="module")
def hk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as m

    return m


def at(a, off=0):
    """`a` on the GPU at a pointer `off` bytes past 256-byte alignment, NaN bit patterns (0xff) around it."""
    raw = np.ascontiguousarray(a).view(np.uint8).reshape(-1)
    buf = torch.full((raw.size + 1024,), 255, dtype=torch.uint8, device="cuda")
    buf[256 + off:256 + off + raw.size] = torch.from_numpy(raw).cuda()
    return buf[256 + off:256 + off + raw.size]


def forced(plan, shares, ops, M, N, K, fa=2, fb=2, la=0, lb=0, f32=1, off_c=0):
    """One call with the plan forced (the measurement build); C between guard values."""
    P = _lib.probes()
    P.mxfp6_probe_slice.argtypes, P.mxfp6_probe_slice.restype = [ctypes.c_int], ctypes.c_int
    guard = torch.full((M * N + 64,), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
    C = guard[16 + off_c:16 + off_c + M * N]
    ta, tb, waves = plan
    prev = P.mxfp6_probe_slice(ta | tb << 4 | waves << 8 | shares << 12)
    try:
        rc = P.mxfp6_gemm_ex(*(ctypes.c_void_p(t.data_ptr()) for t in (*ops, C)), M, N, K, fa, fb, la, lb, f32, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    finally:
        P.mxfp6_probe_slice(prev)
    torch.cuda.synchronize()
    assert rc == 0 and bool((guard[:16 + off_c] == 7.0).all()) and bool((guard[16 + off_c + M * N:] == 7.0).all())
    return C.view(M, N)


@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("M,N,K,la,lb,shares", [(1, 1, 32, 0, 0, 1), (33, 65, 96, 0, 0, 1), (31, 33, 7904, 0, 0, 16), (64, 64, 256, 1, 1, 1), (96, 160, 1152, 1, 0, 2), (128, 96, 2176, 0, 1, 3),
                                                (257, 255, 1056, 0, 0, 2), (17, 260, 384, 0, 0, 1), (32, 32, 6272, 1, 1, 7), (65, 8, 2080, 0, 0, 5)])
def test_plans_vs_oracle(hk, plan, M, N, K, la, lb, shares):
    fa, fb = ((2, 2), (3, 2), (2, 3))[(M + N) % 3]
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(M + K)), fa)
    bp, bsc = co.quantise(o.make_source("weights_outliers", (N, K), np.random.default_rng(N + K)), fb)
    ref = o.gemm_ref(ap, bp, asc, bsc, fa, fb, acc=np.float64)
    a, b = (o.tile_operand(ap), o.tile_scales(asc)) if la else (ap, asc), (o.tile_operand(bp), o.tile_scales(bsc)) if lb else (bp, bsc)
    ops = [at(a[0]), at(b[0]), at(a[1]), at(b[1])]
    got = forced(plan, shares, ops, M, N, K, fa, fb, la, lb).cpu().numpy()
    assert np.isfinite(got).all() and o.rel_err(got, ref) <= 1e-5
    again = forced(plan, shares, ops, M, N, K, fa, fb, la, lb).cpu().numpy()
    assert np.array_equal(got, again)  # added in share order whoever adds; the counters are back at zero
    c16 = forced(plan, shares, ops, M, N, K, fa, fb, la, lb, f32=0)
    assert np.array_equal(c16.view(torch.int16).cpu().numpy().view(np.uint16), o.f32_to_bf16_bits(got))


@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("oa,ob,osa,osb,oc", [(4, 12, 1, 2, 3), (8, 4, 3, 1, 1), (0, 0, 2, 3, 2)])
def test_alignments(hk, plan, oa, ob, osa, osb, oc):
    M, N, K = 70, 136, 608
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(1)), 2)
    bp, bsc = co.quantise(o.make_source("weights", (N, K), np.random.default_rng(2)), 2)
    got = forced(plan, 1, [at(ap, oa), at(bp, ob), at(asc, osa), at(bsc, osb)], M, N, K, off_c=oc).cpu().numpy()
    assert o.rel_err(got, o.gemm_ref(ap, bp, asc, bsc, acc=np.float64)) <= 1e-5


@pytest.mark.parametrize("M,N,K,lb", [(256, 1024, 1024, 1), (128, 512, 2560, 0), (3, 3072, 2688, 0), (48, 704, 928, 0), (90, 390, 3424, 0), (200, 1056, 5120, 1)])
def test_automatic_route(hk, route, M, N, K, lb):
    """Shapes the choice gives to this kernel: fp32, bf16, fused and MXFP6 output on the automatic path, the last one bit for bit
    the quantiser's of the fp32 output."""
    tk = hk.tk_kernel
    assert tk.kernel_choice(M, N, K, 0, lb) in (tk.KERNEL_BLOCK, tk.CHOICE_BLOCK_K_SPLIT)
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(M)), 2)
    bp, bsc = co.quantise(o.make_source("weights", (N, K), np.random.default_rng(N)), 3)
    a, asd, b, bsd = (torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (ap, asc, o.tile_operand(bp) if lb else bp, o.tile_scales(bsc) if lb else bsc))
    got = torch.empty(M, N, device="cuda")
    assert route.gemm(a, b, asd, bsd, got, M, N, K, 2, 3, 0, lb) & 0xff == route.SLICE
    hk.dispatch_micro(a, b, asd, bsd, got, 2, 3, layout_b=lb)
    assert o.rel_err(got.cpu().numpy(), o.gemm_ref(ap, bp, asc, bsc, 2, 3, acc=np.float64)) <= 1e-5
    bias = torch.randn(N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    fused = torch.empty(M, N, device="cuda")
    hk.dispatch_micro(a, b, asd, bsd, fused, 2, 3, layout_b=lb, bias=bias, activation="relu")
    assert torch.equal(fused, (got + bias).clamp_min(0))  # one fp32 addition: exact to its rounding
    if N % 32 == 0:
        cp, cs = torch.empty(M, N // 4 * 3, dtype=torch.uint8, device="cuda"), torch.empty(M, N // 32, dtype=torch.uint8, device="cuda")
        assert route.gemm(a, b, asd, bsd, cp, M, N, K, 2, 3, 0, lb, C_scale=cs) & 0xff == route.SLICE
        hk.dispatch_micro(a, b, asd, bsd, cp, 2, 3, layout_b=lb, C_scale=cs)
        qp, qs = hk.quantize(got, 2)
        assert torch.equal(cp, qp) and torch.equal(cs, qs)


def test_capture_and_streams(hk, route):
    """A K split of this kernel: under capture it runs unsplit, on a stream that has a workspace too; replays equal the eager call (these
    sums are exact)."""
    M, N, K = 64, 512, 12288 + 128
    tk = hk.tk_kernel
    assert tk.kernel_choice(M, N, K) == tk.CHOICE_BLOCK_K_SPLIT
    g = torch.Generator(device="cuda").manual_seed(4)
    (a, asc), (b, bsc) = hk.quantize(torch.randn(M, K, device="cuda", generator=g)), hk.quantize(torch.randn(N, K, device="cuda", generator=g) * 0.02)
    eager = torch.empty(M, N, device="cuda")
    assert route.gemm(a, b, asc, bsc, eager, M, N, K) == route.SLICE | route.SPLIT
    hk.dispatch_micro(a, b, asc, bsc, eager)
    torch.cuda.synchronize()
    for warm in (False, True):
        side, C, graph = torch.cuda.Stream(), torch.zeros(M, N, device="cuda"), torch.cuda.CUDAGraph()
        side.wait_stream(torch.cuda.current_stream())
        if warm:
            with torch.cuda.stream(side):
                hk.dispatch_micro(a, b, asc, bsc, C)
            side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            hk.dispatch_micro(a, b, asc, bsc, C)
        for _ in range(3):
            C.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(C, eager) if warm else o.rel_err(C.cpu().numpy(), eager.cpu().numpy()) <= 1e-5
            hk.dispatch_micro(a, b, asc, bsc, torch.empty_like(C))
            torch.cuda.synchronize()


def order_shows(g, rows, K, scale, sign):
    """Rows whose products with those of the other sign cancel in every other K-block of the first half, 2^18 times the rest: what the
    fp32 sums keep of the rest depends on their order."""
    x = (torch.randn(rows, K, device="cuda", generator=g) * scale).view(rows, K // 32, 32)
    q = K // 128
    x[:, :q:2] *= 2.0**18 if sign < 0 else 1.0
    x[:, q:2 * q:2] = sign * x[:, :q:2]
    return x.reshape(rows, K)


@pytest.mark.parametrize("kind,M,N,K,lb", [("linear", 16, 512, 7680, 1), ("linear", 8, 1024, 8192, 1), ("gemm", 64, 1024, 8192, 0), ("gemm", 16, 512, 15872, 1), ("fp6", 64, 1024, 8192, 0)])
def test_graphs_of_one_stream_share_no_partial_sums(hk, route, kind, M, N, K, lb):
    """Calls whose eager form splits K, captured twice on a stream that has run them: a graph has the bits of one captured on a stream
    that has no workspace (which runs unsplit), not those of the split, alone and replayed beside the other graph and the eager call."""
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = order_shows(g, N, K, 0.02, 1.0)
    xs = [order_shows(g, M, K, 1.0, -1.0) for _ in range(2)]
    if kind == "linear":
        layer = MXFP6Linear(w)
        xs = [x.to(torch.bfloat16) for x in xs]
        call = lambda x: (layer(x),)
        assert route.linear(xs[0], layer, torch.empty(M, N, dtype=torch.bfloat16, device="cuda")) == route.SLICE | route.X | route.SPLIT
    else:
        b, bsc = hk.quantize(w, 2, lb)
        xs = [hk.quantize(x, 2) for x in xs]
        assert route.gemm(xs[0][0], b, xs[0][1], bsc, torch.empty(M, N, device="cuda"), M, N, K, lb=lb) == route.SLICE | route.SPLIT

        def call(x):
            if kind == "gemm":
                C = torch.empty(M, N, device="cuda")
                hk.dispatch_micro(x[0], b, x[1], bsc, C, layout_b=lb)
                return (C,)
            C, S = torch.empty(M, N // 4 * 3, dtype=torch.uint8, device="cuda"), torch.empty(M, N // 32, dtype=torch.uint8, device="cuda")
            hk.dispatch_micro(x[0], b, x[1], bsc, C, layout_b=lb, C_scale=S)
            return C, S

    def captured(x, stream):
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            y = call(x)
        return graph, y

    def copies(stream):
        out = []
        for graph, y in (captured(x, stream) for x in xs):
            graph.replay()
            torch.cuda.synchronize()
            out.append((graph, y, [t.clone() for t in y]))
        return out

    same = lambda y, z: all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(y, z))
    unsplit = [want for _, _, want in copies(torch.cuda.Stream())]
    capture, streams = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    with torch.cuda.stream(capture):
        eager = [call(x) for x in xs]
    torch.cuda.synchronize()
    assert not any(same(y, z) for y, z in zip(eager, unsplit))  # these sums show their order
    graphs = copies(capture)
    assert all(same(want, z) for (_, _, want), z in zip(graphs, unsplit))
    for _ in range(20):
        for s, (graph, _, _) in zip(streams, graphs):
            with torch.cuda.stream(s):
                graph.replay()
        with torch.cuda.stream(capture):
            again = call(xs[0])
        torch.cuda.synchronize()
        assert same(again, eager[0]) and all(same(y, want) for _, y, want in graphs)


# (rows of activations, rows of B / 32, waves) of the instantiations that quantise the activations themselves
X_PLANS = {1: [(8, 1, 4), (8, 1, 8), (8, 2, 4), (8, 2, 8), (16, 1, 4), (16, 1, 8), (16, 2, 4), (16, 2, 6), (32, 1, 4), (32, 2, 4)],
           0: [(8, 1, 4), (8, 1, 8), (8, 2, 4), (8, 2, 6), (16, 1, 4), (16, 2, 4), (24, 1, 4)]}


@pytest.mark.parametrize("bf16,plan", [(b, p) for b in X_PLANS for p in X_PLANS[b]])
@pytest.mark.parametrize("M,N,K,lb,shares", [(1, 1, 32, 0, 1), (7, 65, 96, 0, 1), (33, 33, 7904, 0, 8), (24, 64, 256, 1, 1), (25, 160, 1152, 1, 2), (50, 260, 416, 0, 1), (65, 32, 6272, 1, 5)])
def test_quantising_plans_vs_oracle(hk, bf16, plan, M, N, K, lb, shares):
    """The activations quantised in the kernel: quantiser and product of the oracle.  The output is bf16: half a last place, 2^-8 of
    the value, and the fp32 sums' own bound."""
    P = _lib.probes()
    P.mxfp6_probe_slice.argtypes, P.mxfp6_probe_slice.restype = [ctypes.c_int], ctypes.c_int
    fa, fb = ((2, 2), (3, 2), (2, 3))[(M + N) % 3]
    xs = torch.from_numpy(o.make_source("normal", (M, K), np.random.default_rng(M + K)).astype(np.float32))
    xs[M // 2, :32] = 0  # a block of zeros
    x = xs.to(torch.bfloat16) if bf16 else xs
    ap, asc = co.quantise(x.float().numpy(), fa)
    bp, bsc = co.quantise(o.make_source("weights_outliers", (N, K), np.random.default_rng(N + K)), fb)
    ref = o.gemm_ref(ap, bp, asc, bsc, fa, fb, acc=np.float64)
    ops = [at((x.view(torch.int16) if bf16 else x).numpy()), at(o.tile_operand(bp) if lb else bp), at(o.tile_scales(bsc) if lb else bsc)]
    guard = torch.full((M * N + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    C = guard[16:16 + M * N]
    prev = P.mxfp6_probe_slice(1 | plan[1] << 4 | plan[2] << 8 | shares << 12 | plan[0] << 20)
    try:
        rc = P.mxfp6_linear(ops[0].data_ptr(), bf16, ops[1].data_ptr(), ops[2].data_ptr(), C.data_ptr(), M, N, K, fa, fb, lb, None, 0, 0,
                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    finally:
        P.mxfp6_probe_slice(prev)
    torch.cuda.synchronize()
    assert rc == 0 and bool((guard[:16] == 7.0).all()) and bool((guard[16 + M * N:] == 7.0).all())
    got = C.view(M, N).float().cpu().numpy()
    bound = np.abs(ref) * 2.0**-8 + 1e-5 * np.maximum(np.abs(ref), 0.01 * np.sqrt((ref**2).mean()))
    assert np.isfinite(got).all() and (np.abs(got - ref) <= bound).all()


@pytest.mark.parametrize("M,N,K,bf16", [(5, 512, 1024, 1), (23, 1056, 2080, 1), (64, 512, 1536, 1), (17, 768, 640, 0), (100, 512, 768, 0), (8, 512, 18176, 1), (12, 1024, 1024, 1)])
def test_quantising_route(hk, route, M, N, K, bf16):
    """MXFP6Linear's calls of few rows: the bits of quantise, then GEMM (these sums are exact or rounded far below bf16), eager and
    captured on a stream that has no workspace, odd values in the activations among them.  All but five bf16 rows with K % 512 == 0, which
    stay with the quantiser, run on the slice kernel."""
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(M)
    layer = MXFP6Linear(torch.randn(N, K, device="cuda", generator=g) * 0.02, bias=torch.randn(N, device="cuda", generator=g), activation="relu")
    x = torch.randn(M, K, device="cuda", generator=g)
    x[0, :6] = torch.tensor([float("nan"), float("inf"), -float("inf"), 1e-42, 3e38, -0.0], device="cuda")
    x[M - 1, 64:96] = 1e-41
    x = x.to(torch.bfloat16) if bf16 else x

    def steps():
        xp, xs = hk.quantize(x, 2)
        want = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        hk.dispatch_micro(xp, layer.weight_packed, xs, layer.weight_scale, want, layout_b=layer.layout_w, bias=layer.bias, activation="relu")
        return want

    taken = route.linear(x, layer, torch.empty(M, N, dtype=torch.bfloat16, device="cuda"))
    assert (taken & ~route.SPLIT == route.SLICE | route.X) == ((M, bf16) != (5, 1)) and bool(taken & route.X) == ((M, bf16) != (5, 1))
    assert torch.equal(layer(x).view(torch.int16), steps().view(torch.int16))
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        y = layer(x)
    for _ in range(3):
        x.copy_(torch.randn(M, K, device="cuda", generator=g))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, steps()) and torch.equal(layer(x), steps())


@pytest.mark.parametrize("M,N,K,bf16", [(8, 512, 4096, 1), (16, 512, 7680, 1), (33, 96, 2080, 1), (100, 512, 768, 0), (7, 1024, 2048, 0), (128, 544, 1056, 1)])
def test_layers_whose_products_cancel(hk, route, M, N, K, bf16):
    """Quantised inside the kernel the sums run in another order than in the two calls: both lie within the fp32 sums' rounding of
    the exact product, half a last place (2^-24 of the largest partial sum, sum |x||w| at most) for each of the K / 32 products of a block
    and the up to 32 partial sums of waves and shares, then half a last place of bf16, 2^-9 of the value (2^-8 with the value's own error)."""
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(M + K)
    w, x = order_shows(g, N, K, 0.02, 1.0), order_shows(g, M, K, 1.0, -1.0)
    x = x.to(torch.bfloat16) if bf16 else x
    layer = MXFP6Linear(w)
    assert route.linear(x, layer, torch.empty(M, N, dtype=torch.bfloat16, device="cuda")) & ~route.SPLIT == route.SLICE | route.X
    xp, xs = hk.quantize(x, 2)
    two = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    hk.dispatch_micro(xp, layer.weight_packed, xs, layer.weight_scale, two, layout_b=layer.layout_w)
    wp, ws = co.quantise(w.cpu().numpy(), 2)
    xd, wd = o.dequantise(xp.cpu().numpy(), xs.cpu().numpy(), 2, np.float64), o.dequantise(wp, ws, 2, np.float64)
    ref = xd @ wd.T
    bound = (K / 32 + 32) * 2.0**-24 * (np.abs(xd) @ np.abs(wd).T) + np.abs(ref) * 2.0**-8
    for y in (layer(x), two):
        assert (np.abs(y.float().cpu().numpy() - ref) <= bound).all()
