"""The handle that add_hook leaves: removed, used as a context manager and copied like those of torch's hooks, by a layer
and by a fused block."""
import copy
import io

import pytest
import torch

from tests.test_gpu_layer_attributes import _layer
from tests.util import randn_bf16

pytestmark = pytest.mark.gpu


def _pass(module, K, seed=1):
    x = randn_bf16((32, K), seed).cuda().requires_grad_(True)
    y = module(x)
    y.backward(torch.ones_like(y))
    assert x.grad is not None


@pytest.mark.parametrize("kind", ["w4", "w8", "qat"])
def test_layer(kind):
    from latentq_llm_amd import quant as Q
    m = _layer(kind)
    m.add_hook()
    assert isinstance(m.hook_handle, torch.utils.hooks.RemovableHandle)
    with m.hook_handle as handle:
        assert handle is m.hook_handle
        _pass(m, 512)
        first = m.weight.grad
        assert first is not None and not Q.dict_temp
        first = first.get_value().clone() if isinstance(first, Q.GradientQTensor) else first.clone()
    _pass(m, 512)
    g = m.weight.grad
    assert torch.equal(g.get_value() if isinstance(g, Q.GradientQTensor) else g, first)
    assert len(Q.dict_temp) == 1  # not delivered
    Q.dict_temp.clear()
    m.add_hook()
    _pass(m, 512)
    assert not Q.dict_temp


def test_copies_deliver_to_themselves():
    from latentq_llm_amd import quant as Q
    m = _layer("w4")
    m.add_hook()
    buf = io.BytesIO()
    torch.save(m, buf)
    buf.seek(0)
    for twin in (copy.deepcopy(m), torch.load(buf, weights_only=False)):
        twin.hook_handle.remove()
        _pass(m, 512)
        assert m.weight.grad is not None and getattr(twin.weight, "grad", None) is None and not Q.dict_temp
        twin.add_hook()
        _pass(twin, 512)
        assert twin.weight.grad is not None


def test_block():
    from latentq_llm_amd import quant as Q
    from latentq_llm_amd.fused_mlp import QuantLlamaMLP
    gate, up, down = _layer("w4", 256, 512), _layer("w4", 256, 512), _layer("w4", 512, 256)
    gate.bias = up.bias = None
    block = QuantLlamaMLP(gate, down, up)
    for layer in (gate, up, down):
        layer.add_hook()
    up.hook_handle.remove()
    _pass(block, 512)
    assert gate.weight.grad is not None and down.weight.grad is not None and getattr(up.weight, "grad", None) is None and not Q.dict_temp
