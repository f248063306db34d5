import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def golden_dir():
    return os.path.join(ROOT, "tests", "golden")


class Route:
    """Which kernel the measurement build (the same sources as the operator) runs a call on: mxfp6_probe_route.  Only this thread's
    settings of the measurement build count; kernel and k_split are set for the call."""

    TILED, SKINNY, BLOCK, RING, SLICE = 2, 3, 22, 28, 29
    COPY_A, COPY_B, SPLIT, X = 0x100, 0x200, 0x400, 0x800
    PIECES, KEPT, OUT, STREAM_B = 0, 1, 2, 4  # memory: how the tiled or block kernel of the last call stored C and read B (mxfp6_probe_memory)
    memory = 0

    def _run(self, kernel, k_split, call):
        import torch

        from hipkittensp_amd import _lib

        P = _lib.probes()
        prev = P.mxfp6_set_kernel(kernel), P.mxfp6_set_k_split(k_split)
        try:
            assert call(P, torch.cuda.current_stream().cuda_stream) == 0
            self.memory = P.mxfp6_probe_memory()
            return P.mxfp6_probe_route()
        finally:
            P.mxfp6_set_kernel(prev[0]), P.mxfp6_set_k_split(prev[1])

    def gemm(self, a, b, asc, bsc, C, M, N, K, fa=2, fb=2, la=0, lb=0, C_scale=None, kernel=0, k_split=0):
        import torch

        p = [t.data_ptr() for t in (a, b, asc, bsc, C)]
        if C_scale is not None:
            return self._run(kernel, k_split, lambda P, s: P.mxfp6_gemm_fused_fp6(*p, C_scale.data_ptr(), M, N, K, fa, fb, la, lb, 2, None, 0, None, None, 0, s))
        return self._run(kernel, k_split, lambda P, s: P.mxfp6_gemm_ex(*p, M, N, K, fa, fb, la, lb, int(C.dtype == torch.float32), s))

    def linear(self, x, layer, C):
        import torch

        M, K = x.shape
        N, bias = layer.out_features, layer.bias
        return self._run(0, 0, lambda P, s: P.mxfp6_linear(x.data_ptr(), int(x.dtype == torch.bfloat16), layer.weight_packed.data_ptr(), layer.weight_scale.data_ptr(),
                                                             C.data_ptr(), M, N, K, layer.fmt_x, layer.fmt_w, layer.layout_w, None if bias is None else bias.data_ptr(),
                                                             int(bias is not None and bias.dtype == torch.bfloat16), 0, s))


@pytest.fixture(scope="session")
def route():
    return Route()
