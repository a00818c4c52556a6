"""What watches a call from outside - a trace, a forward-mode level, a function transform - sees a layer as it always did,
although inference without gradients runs the kernels without an autograd Function and training avoids setup_context."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD

from tests.util import make_w4

pytestmark = pytest.mark.gpu
N, K = 256, 512


def w4():
    from latentq_llm_amd import quant as Q
    _, p, s, z = make_w4(N, K, 1)
    m = Q.QLinearA16W4(K, N, bias=False, lbit=0)
    m.zeros.data, m.scales.data, m.wshape = z.clone().cuda(), s.clone().cuda(), [N, K]
    m.weight.set_value(p.cuda(), [m.scales, m.zeros, m.wshape])
    return m


def w8():
    from latentq_llm_amd import quant as Q
    m = Q.QLinearA8W8(K, N, bias=False)
    m.qscales.data = torch.full((N, 1), 2e-3, dtype=torch.bfloat16, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(1)
    m.weight.set_value(torch.randint(-127, 128, (N, K), device="cuda", dtype=torch.int8, generator=gen), m.qscales)
    return m


def rows(seed, m=3):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(m, K, device="cuda", generator=gen).to(torch.bfloat16)


@pytest.mark.parametrize("make", [w4, w8])
@pytest.mark.parametrize("grad", [False, True])
def test_a_trace_follows_its_input(make, grad):
    m, x, other = make(), rows(1), rows(2)
    with torch.set_grad_enabled(grad):
        t = torch.jit.trace(lambda v: m(v) * 1, x, check_trace=False)
        assert torch.equal(t(other), m(other)) and not torch.equal(m(x), m(other))


@pytest.mark.parametrize("make", [w4, w8])
@pytest.mark.parametrize("grad", [False, True])
def test_forward_mode_is_refused(make, grad):
    m, x = make(), rows(1)
    with fwAD.dual_level(), torch.set_grad_enabled(grad), pytest.raises(NotImplementedError):
        m(fwAD.make_dual(x, torch.ones_like(x)))


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("grad", [False, True])
def test_functional_gradient_around_a_layer(train, grad):
    m, x = w4(), rows(1)
    want = m(x).float().sum()
    if train:
        m.weight.requires_grad = True
        m.add_hook()
    with torch.set_grad_enabled(grad):
        got = torch.func.grad(lambda s: (m(x).float() * s).sum())(torch.tensor(2.0, device="cuda"))
    assert torch.allclose(got, want)


@pytest.mark.parametrize("make", [w4, w8])
@pytest.mark.parametrize("grad", [False, True])
def test_vmap_is_refused(make, grad):
    m, x = make(), rows(1)
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError):
        torch.func.vmap(lambda v: m(v))(x.view(3, 1, K))


def test_wrapped_tensors_do_not_reach_the_kernels():
    """The binding takes memory, not wrappers that look like plain tensors."""
    from latentq_llm_amd import ops
    m, x = w4(), rows(1)
    w = (m.weight.data, m.scales, m.zeros, (N, K))
    assert torch.func.vmap(lambda v: torch.tensor(ops.linear4(v, *w) is None, device="cuda"), out_dims=None)(x.view(3, 1, K))
