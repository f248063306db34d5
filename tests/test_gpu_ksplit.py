"""The K split's partial sums (accumulator order, common.hpp partial_offset) and their reduction at the edges of its 32 x 32 tiles
and of its unrolling over the shares, against the CPU oracle.  Bound: as in test_gpu_ragged.py -- fp32 sums held to 1e-5 of the
oracle's, bf16 the rounding of the fp32 result bit for bit, a bias one fp32 addition."""
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


def call(hk, ops, M, N, dtype, kernel, shares, **kw):
    guard = torch.full((M * N + 64,), 7.0, dtype=dtype, device="cuda")
    C = guard[32:32 + M * N].view(M, N)
    pk, ps = hk.tk_kernel.set_kernel(kernel), hk.tk_kernel.set_k_split(shares)
    try:
        hk.dispatch_micro(*ops, C, 2, 2, **kw)
        torch.cuda.synchronize()
    finally:
        hk.tk_kernel.set_kernel(pk)
        hk.tk_kernel.set_k_split(ps)
    assert bool((guard[:32] == 7.0).all()) and bool((guard[32 + M * N:] == 7.0).all())
    return C


@pytest.mark.parametrize("M,N", [(1, 8), (32, 32), (33, 40), (127, 136), (129, 264)])
@pytest.mark.parametrize("kernel,shares", [(22, 2), (22, 3), (22, 4), (22, 5), (22, 6), (22, 8), (22, 9), (6, 2), (5, 3)])
def test_partial_sums_and_reduction_vs_oracle(hk, M, N, kernel, shares):
    K = 1024 * shares
    ap, asc = co.quantise(o.make_source("normal", (M, K), np.random.default_rng(M + shares)), 2)
    bp, bsc = co.quantise(o.make_source("weights", (N, K), np.random.default_rng(N + shares)), 2)
    ops = [torch.from_numpy(x).cuda() for x in (ap, bp, asc, bsc)]
    got = call(hk, ops, M, N, torch.float32, kernel, shares).cpu().numpy()
    assert np.isfinite(got).all() and o.rel_err(got, o.gemm_ref(ap, bp, asc, bsc, acc=np.float64)) <= 1e-5
    c16 = call(hk, ops, M, N, torch.bfloat16, kernel, shares)
    assert np.array_equal(c16.view(torch.int16).cpu().numpy().view(np.uint16), o.f32_to_bf16_bits(got))
    bias = torch.randn(N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    fused = call(hk, ops, M, N, torch.float32, kernel, shares, bias=bias, activation="relu").cpu().numpy()
    assert np.array_equal(fused, np.maximum(got + bias.cpu().numpy(), 0).astype(np.float32))
