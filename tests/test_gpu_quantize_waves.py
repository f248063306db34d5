"""The quantiser's launch of one wave per workgroup (up to 1024 chunks of 64 blocks) against that of four, bit for bit: a matrix past the
line and its halves below it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,K", [(1024, 2048), (1152, 2048), (2176, 1152), (4096, 640)])
def test_halves_match_the_whole(rows, K, dtype, layout):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import hipkittensp_amd as hk

    g = torch.Generator(device="cuda").manual_seed(rows)
    X = (torch.randn(rows, K, device="cuda", generator=g) * torch.exp2(torch.randint(-9, 9, (rows, 1), device="cuda", generator=g).float())).to(dtype)
    for fmt in (2, 3):
        whole = hk.quantize(X, fmt, layout)
        parts = [hk.quantize(x.contiguous(), fmt, layout) for x in X.view(4, rows // 4, K)]
        for i in range(2):
            assert torch.equal(whole[i], torch.cat([p[i] for p in parts]))
