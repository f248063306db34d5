"""What this library's users have it do, as cases that can be timed: GEMMs on packed MXFP6 operands
(tk_kernel.dispatch_micro), linear layers on bf16 or fp32 activations (torch_op.MXFP6Linear), a two-layer MLP whose
hidden activations stay MXFP6 (dispatch_micro with C_scale), and the quantisation of weights (tk_kernel.quantize).

A case is a dict of plain values; listed() gives the fixed ones, draw() one more of the same ranges, prepare() what a
program holds before the call, run() one pass, work() the bytes and operations a pass cannot do without and tolerance()
how far another correct implementation's outputs may lie from this one's.
"""
import math

import torch

from hipkittensp_amd import tk_kernel
from hipkittensp_amd.torch_op import MXFP6Linear

E2M3, E3M2 = tk_kernel.E2M3, tk_kernel.E3M2


def _linear(M, N, K, bias=True, act="none", x="bf16"):
    return {"kind": "linear", "M": M, "N": N, "K": K, "bias": bias, "act": act, "x": x}


def _gemm(M, N, K, fmt_a=E2M3, fmt_b=E2M3, tile_a=False, tile_b=False, out="bf16"):
    return {"kind": "gemm", "M": M, "N": N, "K": K, "fmt_a": fmt_a, "fmt_b": fmt_b, "tile_a": tile_a, "tile_b": tile_b, "out": out}


def _mlp(M, K, H, act="silu"):
    return {"kind": "mlp", "M": M, "K": K, "H": H, "act": act}


def _quantize(rows, K, x="fp32", tile=True, fmt=E2M3):
    return {"kind": "quantize", "rows": rows, "K": K, "x": x, "tile": tile, "fmt": fmt}


def listed():
    return [
        # one token through a projection of a model that decodes: the smallest call, latency and launches
        dict(_linear(1, 4096, 4096), name="linear_decode_1"),
        # a batch of requests, as many as there happen to be, through a down projection
        dict(_linear(23, 4096, 14336), name="linear_decode_23"),
        # a prompt of a few thousand tokens through an up projection with its activation
        dict(_linear(2048, 14336, 4096, act="silu"), name="linear_prefill"),
        # the smallest GEMM of the benchmark: launch-bound
        dict(_gemm(256, 256, 256), name="gemm_256"),
        # decode against a wide weight matrix as the quantiser leaves it (row-major)
        dict(_gemm(16, 8192, 28672), name="gemm_decode_16"),
        # batched decode against prepared (tile-major) weights
        dict(_gemm(64, 8192, 28672, tile_b=True), name="gemm_decode_64"),
        # a chunk of a prompt, or a large batch, against prepared weights
        dict(_gemm(256, 8192, 28672, tile_b=True), name="gemm_chunk_256"),
        # the headline square, from row-major operands
        dict(_gemm(8192, 8192, 8192), name="gemm_8192"),
        # mixed formats, prepared weights, the longest K: the largest work
        dict(_gemm(8192, 8192, 16384, fmt_a=E3M2, tile_b=True), name="gemm_mixed_16384"),
        # sizes that no tile divides: rows, columns and K-blocks as they come
        dict(_gemm(500, 5003, 2880), name="gemm_ragged"),
        # an MLP block on MXFP6 activations: the first layer's output is the second one's operand
        dict(_mlp(1024, 4096, 14336), name="mlp_1024"),
        # a weight matrix made ready for use: fp32 in, packed operand and scales out in the kernels' order
        dict(_quantize(8192, 28672), name="quantize_weights"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, steps):
    """A size over its logarithm, as a multiple of one of `steps`."""
    step = rng.choice(steps)
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["linear", "linear", "gemm", "gemm", "gemm", "mlp", "quantize"])
    if kind == "quantize":
        tile = rng.random() < 0.6
        rows, K = _width(rng, 256, 8192, [32] if tile else [1, 8]), _width(rng, 512, 28672, [128, 512] if tile else [32, 128])
        return _quantize(rows, K, rng.choice(["fp32", "bf16"]), tile, rng.choice([E2M3, E2M3, E3M2]))
    # every size of model a GPU holds: narrow projections to wide ones; most widths are multiples of 128 or 512, some of
    # less; rows from one token to a long prompt, most of them not a multiple of anything
    while True:
        M = _log(rng, 1, 8192) if rng.random() < 0.6 else 1 << rng.randrange(14)
        if kind == "mlp":
            c = _mlp(M, _width(rng, 1024, 8192, [128, 512]), _width(rng, 2048, 28672, [128, 512]), rng.choice(["relu", "gelu", "silu"]))
            size = 2 * M * c["K"] * c["H"]
        else:
            ragged = rng.random() < 0.25
            N = _width(rng, 256, 28672, [1, 8, 32] if ragged else [128, 512])
            K = _width(rng, 256, 28672, [32] if ragged else [128, 512, 512])
            size = M * N * K
            if kind == "linear":
                c = _linear(M, N, K, rng.random() < 0.5, rng.choice(["none", "none", "gelu", "silu"]), rng.choice(["bf16", "bf16", "fp32"]))
            else:
                tile_b = rng.random() < 0.5 and N % 32 == 0 and K % 128 == 0
                tile_a = tile_b and rng.random() < 0.5 and M % 32 == 0
                fmt_a, fmt_b = rng.choice([(E2M3, E2M3), (E2M3, E2M3), (E3M2, E2M3), (E2M3, E3M2)])
                c = _gemm(M, N, K, fmt_a, fmt_b, tile_a, tile_b, rng.choice(["bf16", "bf16", "bf16", "fp32"]))
        if size <= 8192 * 8192 * 8192:
            return c


def _randn(seed, index, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + index)
    return torch.randn(*shape, generator=g, device="cuda")


def _activations(seed, index, M, K):
    return _randn(seed, index, M, K)


def _weights(seed, index, N, K):
    return _randn(seed, index, N, K).mul_(0.02)


def _layout(tile):
    return tk_kernel.LAYOUT_TILE if tile else tk_kernel.LAYOUT_ROW


def prepare(case, seed):
    if case["kind"] == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        bias = _randn(seed, 2, N).mul_(0.1).to(torch.bfloat16) if case["bias"] else None
        layer = MXFP6Linear(_weights(seed, 1, N, K), bias=bias, activation=case["act"])
        x = _activations(seed, 0, M, K)
        return {"kind": "linear", "layer": layer, "x": x.to(torch.bfloat16) if case["x"] == "bf16" else x}
    if case["kind"] == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        la, lb = _layout(case["tile_a"]), _layout(case["tile_b"])
        A, As = tk_kernel.quantize(_activations(seed, 0, M, K), case["fmt_a"], la)
        B, Bs = tk_kernel.quantize(_weights(seed, 1, N, K), case["fmt_b"], lb)
        C = torch.empty(M, N, dtype=torch.bfloat16 if case["out"] == "bf16" else torch.float32, device="cuda")
        return {"kind": "gemm", "args": (A, B, As, Bs, C, case["fmt_a"], case["fmt_b"], la, lb)}
    if case["kind"] == "mlp":
        M, K, H = case["M"], case["K"], case["H"]
        tile = tk_kernel.LAYOUT_TILE
        X, Xs = tk_kernel.quantize(_activations(seed, 0, M, K))
        W1, W1s = tk_kernel.quantize(_weights(seed, 1, H, K), E2M3, tile)
        W2, W2s = tk_kernel.quantize(_weights(seed, 2, K, H), E2M3, tile)
        Hp = torch.empty(M, H // 4 * 3, dtype=torch.uint8, device="cuda")
        Hs = torch.empty(M, H // 32, dtype=torch.uint8, device="cuda")
        Y = torch.empty(M, K, dtype=torch.bfloat16, device="cuda")
        return {"kind": "mlp", "up": (X, W1, Xs, W1s, Hp, E2M3, E2M3, tk_kernel.LAYOUT_ROW, tile), "act": case["act"], "Hs": Hs,
                "down": (Hp, W2, Hs, W2s, Y, E2M3, E2M3, tk_kernel.LAYOUT_ROW, tile)}
    X = _weights(seed, 0, case["rows"], case["K"])
    return {"kind": "quantize", "args": (X if case["x"] == "fp32" else X.to(torch.bfloat16), case["fmt"], _layout(case["tile"]))}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "gemm":
        tk_kernel.dispatch_micro(*state["args"])
        return state["args"][4]
    if kind == "mlp":
        tk_kernel.dispatch_micro(*state["up"], activation=state["act"], C_scale=state["Hs"])
        tk_kernel.dispatch_micro(*state["down"])
        return state["down"][4]
    return tk_kernel.quantize(*state["args"])


def work(case):
    packed = 0.75 + 1 / 32  # bytes of a packed element and its share of a scale
    if case["kind"] == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": (2 if case["x"] == "bf16" else 4) * M * K + packed * N * K + 2 * M * N + (2 * N if case["bias"] else 0), "flops": 2 * M * N * K}
    if case["kind"] == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": packed * K * (M + N) + (2 if case["out"] == "bf16" else 4) * M * N, "flops": 2 * M * N * K}
    if case["kind"] == "mlp":
        M, K, H = case["M"], case["K"], case["H"]
        return {"bytes": packed * (M * K + 2 * K * H) + 2 * M * K, "flops": 4 * M * K * H}
    return {"bytes": ((4 if case["x"] == "fp32" else 2) + packed) * case["rows"] * case["K"], "flops": 0}


def tolerance(case):
    # Against the same product of the dequantised operands in float64: bf16 results differ in one last place (0.0078 of a
    # value) at 6e-4 of the outputs behind a gelu, 3.3e-5 in norm, and not at all elsewhere; fp32 results not at all (sums
    # of a few thousand products of 4-bit significands are exact, longer ones good to the last place or two).  A hidden
    # activation that another correct sum rounds to its other MXFP6 neighbour moves an output of the MLP by far less
    # than its last place.
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "gemm" and case["out"] == "fp32":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 1.5e-4, "max": 1e-2}
