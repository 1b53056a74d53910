"""BitLinear on fp32 rows in one call (quantize, product, scale, bias) against the
oracle's quantizer and product, bit for bit: widths on both sides of the
quantizer's wave form (multiples of four up to 4096) and of its row sizes, padded
columns, row counts on both sides of the GEMV, with and without a bias; and the
model's float logits against its integer ones."""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 5, 37, 64, 65, 130])
@pytest.mark.parametrize("k,n", [(1, 4), (3, 8), (4, 20), (62, 64), (1000, 132), (1022, 64), (1024, 64), (1028, 36),
                                 (2048, 128), (2052, 4), (4096, 16), (4100, 16)])
@pytest.mark.parametrize("bias", [False, True])
def test_bitlinear_f32(cuda, m, k, n, bias):
    import torch
    from rational_bitnet import BitLinear, weight_quant_ternary
    g = torch.Generator().manual_seed(m * 10007 + k + n)
    layer = BitLinear(k, n, bias=bias)
    with torch.no_grad():
        layer.weight.copy_(torch.randn(n, k, generator=g))
        if bias:
            layer.bias.copy_(torch.randn(n, generator=g))
    x = torch.randn(m, k, generator=g) * torch.logspace(-12, 6, m).unsqueeze(1)
    x[-1] = 0
    q, s = O.act_quant_f32(x.numpy())
    wq, ws = weight_quant_ternary(layer.weight.detach())
    acc = q.astype(np.int64) @ wq.numpy().astype(np.int64).T
    ref = acc.astype(np.float32) * (np.float32(float(ws)) * s)[:, None]
    if bias:
        ref = ref + layer.bias.detach().numpy()
    y = layer.cuda()(x.cuda())
    assert np.array_equal(y.cpu().numpy(), ref)


@pytest.mark.parametrize("vocab", [64, 66])
def test_float_logits(cuda, vocab):
    import torch
    from mamba_integer_model import MambaIntegerModel
    model = MambaIntegerModel({"d_model": 64, "n_layer": 2, "vocab_size": vocab, "ssm_cfg": {"d_state": 16, "dt_rank": 16}})
    for shape in ((1, 3), (2, 70)):
        ids = torch.randint(0, vocab, shape, device="cuda")
        want = model.forward_int(ids).to(torch.float32) * model.logit_scale
        assert torch.equal(model(ids), want)
