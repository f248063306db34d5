"""MXFP6Linear reads its weights straight from the module's buffers: what replaces a buffer counts on the next call."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layers():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from hipkittensp_amd.torch_op import MXFP6Linear

    g = torch.Generator(device="cuda").manual_seed(1)
    made = [MXFP6Linear(torch.randn(256, 512, device="cuda", generator=g), bias=torch.randn(256, device="cuda", generator=g)) for _ in range(2)]
    return made, torch.randn(3, 512, device="cuda", generator=g).to(torch.bfloat16)


def test_replaced_buffers_count(layers):
    (a, b), x = layers
    ya, yb = a(x), b(x)
    assert not torch.equal(ya, yb)
    assert torch.equal(torch.func.functional_call(a, dict(b.named_buffers()), x), yb) and torch.equal(a(x), ya)
    kept = a.weight_packed, a.weight_scale, a.bias
    a.weight_packed, a.weight_scale, a.bias = b.weight_packed, b.weight_scale, b.bias
    assert torch.equal(a(x), yb)
    a.weight_packed, a.weight_scale, a.bias = kept
    a.load_state_dict(a.state_dict())
    assert torch.equal(a(x), ya)


def test_a_parameter_in_a_buffers_place(layers):
    (a, _), x = layers
    ya, w = a(x), a.weight_packed
    del a.weight_packed
    a.weight_packed = torch.nn.Parameter(w, requires_grad=False)
    try:
        assert "weight_packed" not in a._buffers and torch.equal(a(x), ya)
    finally:
        del a.weight_packed
        a.register_buffer("weight_packed", w)
