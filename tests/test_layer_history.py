"""The history that a layer's result gets in training is an autograd Function's: its backward can be captured by compiled autograd, a
layer that keeps its own result is collected, and the node shows what it saved."""
import gc
import weakref

import pytest
import torch

from latentq_llm_amd import quant as Q


class Base(torch.autograd.Function):
    pass


def grads(left, saved, dy, wanted):
    dy = Q._rows(dy)
    left.append(wanted)
    return dy @ saved[1].t() if wanted else None


def result(lead=(3,), bias=True, left=None):
    gen = torch.Generator().manual_seed(1)
    x, w = torch.randn(lead + (4,), generator=gen, requires_grad=True), torch.randn(4, 5, generator=gen)
    b = torch.zeros(5, requires_grad=True) if bias else None
    left = [] if left is None else left
    return x, w, Q._attach(x.detach() @ w, x, b, (x, w), grads, left, Base), left


@pytest.mark.parametrize("lead", [(), (3,), (2, 3)])
@pytest.mark.parametrize("bias", [True, False])
def test_gradient(lead, bias):
    x, w, y, left = result(lead, bias)
    dy = torch.randn(y.shape)
    y.backward(dy)
    assert torch.equal(x.grad, (dy.reshape(-1, 5) @ w.t()).view(x.shape)) and left == [True]


def test_compiled_autograd():
    from torch._dynamo import compiled_autograd
    x, w, y, _ = result()
    captured = []

    def compiler(graph):
        captured.append(graph)
        return graph
    with compiled_autograd._enable(compiler):
        y.backward(torch.ones(3, 5))
    assert captured and torch.allclose(x.grad, w.sum(1).expand(3, 4))


def test_a_layer_that_keeps_its_result_is_collected():
    class Layer:
        calls = ()

        def append(self, wanted):
            self.calls += (wanted,)
    layer = Layer()
    layer.out = result(left=layer)[2]
    gone = weakref.ref(layer)
    del layer
    gc.collect()
    assert gone() is None


def test_what_the_node_shows():
    x, w, y, _ = result()
    assert y.grad_fn.name() == "BaseBackward" and y.grad_fn.needs_input_grad[:2] == (True, True)
    assert y.grad_fn.saved_tensors[0] is x and torch.equal(y.grad_fn.saved_tensors[1], w)
    y.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        y.sum().backward()
