"""A layer in training attaches its backward to its result itself where nothing watches; hooks on saved tensors, among others, send it
through its autograd Function. Both ways give the same outputs and gradients, and refuse the same misuse."""
import pytest
import torch

from tests.util import make_w4

pytestmark = pytest.mark.gpu
N, K = 512, 256


def make(kind, bias=True, gbit=16):
    from latentq_llm_amd import quant as Q
    from latentq_llm_amd.fused_mlp import QuantLlamaMLP

    def w4(n, k, seed, bias):
        _, p, s, z = make_w4(n, k, seed)
        m = Q.QLinearA16W4(k, n, bias=bias, lbit=4, gbit=gbit)
        m.zeros.data, m.scales.data = z.cuda(), s.cuda()
        m.weight.set_value(p.cuda(), [m.scales, m.zeros, m.wshape])
        return m
    gen = torch.Generator(device="cuda").manual_seed(1)
    if kind == "mlp":
        m = QuantLlamaMLP(w4(N, K, 1, False), w4(K, N, 2, bias), w4(N, K, 3, False))
        layers = [m.gate_proj, m.up_proj, m.down_proj]
    elif kind == "w4":
        m = w4(N, K, 1, bias)
        layers = [m]
    else:
        m = Q.QLinearQAT(K, N, bias=bias) if kind == "qat" else Q.QLinearA8W8(K, N, bias=bias, lbit=4, gbit=gbit)
        m.qscales.data = torch.full((N, 1), 2e-3, dtype=torch.bfloat16, device="cuda")
        w8 = torch.randint(-127, 128, (N, K), device="cuda", dtype=torch.int8, generator=gen)
        if kind == "qat":
            m.weight.data = (w8.to(torch.bfloat16) * m.qscales).contiguous()
        else:
            m.act_quant = "per_token" if kind == "w8_token" else "per_tensor"
            m.weight.set_value(w8, m.qscales)
        layers = [m]
    for layer in layers:
        if layer.bias is not None:
            layer.bias.data = torch.randn(layer.output_features, device="cuda", generator=gen).to(torch.bfloat16)
        layer.add_hook()
    return m, layers


def x_of(shape, seed=5):
    return torch.randn(shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)).to(torch.bfloat16)


def through_function():
    return torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t)


def kind_of(y):
    return y.grad_fn.name()


KINDS = ["w4", "w8", "w8_token", "qat", "mlp"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("lead", [(), (3,), (64,), (2, 65), (1, 2, 33)])
@pytest.mark.parametrize("gbit", [16, 8])
def test_same_as_the_function(hip_lib, kind, lead, gbit):
    from latentq_llm_amd.quant import GradientQTensor, dict_temp
    if kind == "qat" and gbit == 8:
        gbit = 16
    got = []
    for function in (False, True):
        GradientQTensor.noise_seed, GradientQTensor._noise_offset = 3, 0
        m, layers = make(kind, gbit=gbit)
        out = []
        for step in (1, 2):
            x = x_of(lead + (K,), step).requires_grad_(True)
            if function:
                with through_function():
                    y = m(x)
            else:
                y = m(x)
            assert y.shape == x.shape[:-1] + (K if kind == "mlp" else N,)
            y.backward(x_of(y.shape, 10 + step))
            out += [y.detach(), x.grad]
        for layer in layers:
            g = layer.weight.grad
            out += [g.qdata, g.scale] if isinstance(g, GradientQTensor) else [g]
            assert layer.bias is None or layer.bias.grad is None
        assert not dict_temp
        got.append(out)
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", KINDS)
def test_what_autograd_asks_of_a_node(hip_lib, kind):
    m, layers = make(kind)
    out = K if kind == "mlp" else N
    x = x_of((4, K)).requires_grad_(True)
    dy = x_of((4, out), 7)
    y = m(x)
    a, = torch.autograd.grad(y, x, dy, retain_graph=True)
    b, = torch.autograd.grad(y, x, dy)
    assert torch.equal(a, b)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, x, dy)
    # rows that come as an expanded number, and a result of no consequence
    x2 = x.detach().clone().requires_grad_(True)
    m(x2).sum().backward()
    x3 = x.detach().clone().requires_grad_(True)
    m(x3).backward(torch.ones(4, out, dtype=torch.bfloat16, device="cuda"))
    assert torch.equal(x2.grad, x3.grad)
    # changed between forward and backward
    x4 = x.detach().clone()
    z = x4.requires_grad_(True) * 1
    y = m(z)
    if kind not in ("w8", "w8_token"):  # (these keep the int8 activations)
        z.detach().add_(1)
        with pytest.raises(RuntimeError, match="inplace"):
            y.backward(dy)
    # hooks of the caller's, on the result and on the node
    x5 = x.detach().clone().requires_grad_(True)
    y = m(x5)
    y.register_hook(lambda g: g * 2)
    seen = []
    y.grad_fn.register_hook(lambda gi, go: seen.append((len(gi), len(go))))
    y.backward(dy)
    x6 = x.detach().clone().requires_grad_(True)
    m(x6).backward(dy * 2)
    assert torch.equal(x5.grad, x6.grad) and seen and seen[0][1] == 1


@pytest.mark.parametrize("kind", ["w4", "w8", "qat"])
def test_weight_gradient_where_only_the_bias_asks_for_one(hip_lib, kind):
    m, layers = make(kind)
    x, dy = x_of((4, K)), x_of((4, N), 7)
    y = m(x)
    assert y.requires_grad  # the bias is a parameter
    y.backward(dy)
    first = m.weight.grad.clone()
    m.weight.grad = None
    with through_function():
        y = m(x)
    y.backward(dy)
    assert torch.equal(first, m.weight.grad)
    twin, _ = make(kind, bias=False)
    assert not twin(x).requires_grad


def test_an_error_in_a_backward_reaches_the_caller(hip_lib, monkeypatch):
    from latentq_llm_amd import quant as Q
    m, _ = make("w4")
    x = x_of((4, K)).requires_grad_(True)
    y = m(x)

    def fails(*a):
        raise ValueError("no such gradient")
    monkeypatch.setattr(Q, "_hand_over", fails)
    with pytest.raises(ValueError, match="no such gradient"):
        y.backward(x_of((4, N), 7))


@pytest.mark.parametrize("kind", ["w4", "w8", "mlp"])
@pytest.mark.parametrize("reentrant", [False, True])
def test_recomputation(hip_lib, kind, reentrant):
    from torch.utils.checkpoint import checkpoint
    m, layers = make(kind)
    dy = x_of((4, K if kind == "mlp" else N), 7)
    grads = []
    for wrapped in (False, True):
        for layer in layers:
            layer.weight.grad = None
        x = x_of((4, K)).requires_grad_(True)
        y = checkpoint(m, x, use_reentrant=reentrant) if wrapped else m(x)
        y.backward(dy)
        grads.append([x.grad] + [layer.weight.grad for layer in layers])
    for a, b in zip(*grads):
        assert torch.equal(a, b)


def test_the_node_is_taken(hip_lib):
    m, _ = make("w4")
    x = x_of((2, 3, K)).requires_grad_(True)
    y = m(x)
    assert kind_of(y) == "QLinearFunctionW4Backward" and len(y.grad_fn.next_functions) == 2
    with through_function():
        assert "View" in kind_of(m(x))  # the Function's rows, shaped again


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("lead", [(4,), (2, 33)])
def test_compiled_autograd(hip_lib, kind, lead):
    """The forward as ever, the backward captured and run as a graph."""
    from torch._dynamo import compiled_autograd
    m, layers = make(kind)
    dy = x_of(lead + (K if kind == "mlp" else N,), 7)
    grads = []
    for captured in (False, True):
        for layer in layers:
            layer.weight.grad = None
        x = x_of(lead + (K,)).requires_grad_(True)
        y = m(x)
        if captured:
            with compiled_autograd._enable(lambda graph: graph):
                y.backward(dy)
        else:
            y.backward(dy)
        grads.append([x.grad] + [layer.weight.grad for layer in layers])
    for a, b in zip(*grads):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", KINDS)
def test_a_layer_that_keeps_its_result_is_collected(hip_lib, kind):
    import gc
    import weakref
    m, layers = make(kind)
    m.out = m(x_of((4, K)).requires_grad_(True))
    gone = weakref.ref(m)
    del m, layers
    gc.collect()
    assert gone() is None
