"""Layers in inference whose bias or scales are not where the constructor put them: a parametrised bias, and plain
attributes as replicating and sharding wrappers leave them."""
import pytest
import torch
import torch.nn as nn
from torch.nn.utils import parametrize

from tests.util import make_w4, randn_bf16

pytestmark = pytest.mark.gpu


def _layer(kind, N=256, K=512):
    from latentq_llm_amd import quant as Q
    if kind == "w4":
        m = Q.QLinearA16W4(K, N, bias=True)
        _, p, s, z = make_w4(N, K, 1)
        m.scales.data, m.zeros.data = s.cuda(), z.cuda()
        m.weight.set_value(p.cuda(), [m.scales, m.zeros, m.wshape])
    else:
        m = Q.QLinearA8W8(K, N, bias=True) if kind == "w8" else Q.QLinearQAT(K, N, bias=True)
        m.qscales.data = (randn_bf16((N, 1), 2).abs() * 1e-3 + 1e-4).cuda()
        if kind == "w8":
            m.weight.set_value(torch.randint(-127, 128, (N, K), generator=torch.Generator().manual_seed(3), dtype=torch.int8).cuda(), m.qscales)
        else:
            m.weight.data = randn_bf16((N, K), 4, 0.05).cuda()
    m.bias.data = randn_bf16((N,), 5).cuda()
    return m


@pytest.mark.parametrize("kind", ["w4", "w8", "qat"])
@pytest.mark.parametrize("M", [1, 40])
def test_bias_and_scales_elsewhere(kind, M):
    class Doubled(nn.Module):
        def forward(self, b):
            return 2 * b

    x = randn_bf16((M, 512), 6).cuda()
    plain = _layer(kind)
    with torch.no_grad():
        want = plain(x)
        m = _layer(kind)
        m.bias.data = (m.bias.data / 2).contiguous()
        parametrize.register_parametrization(m, "bias", Doubled())
        assert torch.equal(m(x), want)
        m = _layer(kind)
        bias = m.bias.data
        del m.bias
        m.bias = bias
        if kind != "w4":
            scales = m.qscales.data
            del m.qscales
            m.qscales = scales
        assert torch.equal(m(x), want)


@pytest.mark.parametrize("kind", ["w4", "w8"])
@pytest.mark.parametrize("M", [1, 40])
def test_bias_as_constructed(kind, M, monkeypatch):
    """A bias in fp32, as the constructor leaves it, is rounded to bf16 and takes the direct path too."""
    x = randn_bf16((M, 512), 6).cuda()
    m = _layer(kind)
    m.bias.data = m.bias.data.float() * 1.001
    want = m(x).detach()  # through the Function
    monkeypatch.setattr(type(m), "_apply_fn", None)
    with torch.no_grad():
        assert m.bias.dtype == torch.float32 and torch.equal(m(x), want)
