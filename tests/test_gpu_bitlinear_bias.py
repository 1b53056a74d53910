"""BitLinear's bias: the shapes that torch's broadcasting adds to the product."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(12,), (1,), (), (1, 12), (5, 12), (5, 1)])
def test_bias_shapes(cuda, shape):
    import torch
    from rational_bitnet import BitLinear
    torch.manual_seed(0)
    layer, plain = BitLinear(40, 12, bias=True).to(cuda), BitLinear(40, 12).to(cuda)
    plain.weight = layer.weight
    layer.bias = torch.nn.Parameter(torch.randn(shape, device=cuda))
    x = torch.randn(5, 40, device=cuda)
    assert torch.equal(layer(x), plain(x) + layer.bias)
