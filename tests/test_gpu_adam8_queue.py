"""What waits inside MyAdam.step(): a replaced update_step sees every parameter's step finished, a launch that fails leaves
the parameters and their gradients, waiting steps keep a bounded amount of memory, and a parameter listed twice takes
one step."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _weights(latent, shapes, gbit=16):
    from latentq_llm_amd import quant as Q
    gen = torch.Generator(device="cuda").manual_seed(1)
    out = []
    for n, k in shapes:
        groups = n * k // 128
        if latent == "w8":
            m = Q.QLinearA8W8(k, n, bias=False, lbit=4, gbit=gbit)
            m.qscales.data = (torch.rand((n, 1), generator=gen, device="cuda") * 1e-3 + 1e-4).to(torch.bfloat16)
            m.weight.set_value(torch.randint(-127, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8), m.qscales)
        else:
            m = Q.QLinearA16W4(k, n, bias=False, lbit=0 if latent == "sr" else 4, gbit=gbit)
            m.scales.data = (torch.rand((groups, 1), generator=gen, device="cuda") * 0.01 + 1e-3).to(torch.bfloat16)
            m.zeros.data = torch.randint(6, 10, (groups, 1), generator=gen, device="cuda").to(torch.bfloat16)
            m.weight.set_value(torch.randint(-128, 128, (n * k // 2,), generator=gen, device="cuda", dtype=torch.int8), [m.scales, m.zeros, m.wshape])
        out.append(m.weight)
    return out


def _grads(weights, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    for w in weights:
        w.grad = (torch.randn(tuple(w.shape), generator=gen, device="cuda") * 1e-2).to(torch.bfloat16)


def _adam(weights, cls=None):
    from latentq_llm_amd import quant as Q
    return (cls or Q.MyAdam)([{"params": weights}], lr=1e-3, betas=(0.9, 0.95), obit=8, sr_seed=5)


def _seen(opt, w):
    s = opt.state[w]
    return [w.data.clone(), w.grad] + [s[k].clone() for k in ("state1", "qmap1", "absmax1", "state2", "qmap2", "absmax2")] + (
        [w.residual.residual_int.clone()] if w.residual is not None else [])


@pytest.mark.parametrize("how", ["subclass", "instance", "class"])
@pytest.mark.parametrize("latent", ["sr", "w4", "w8"])
def test_a_replaced_update_step_sees_finished_steps(hip_lib, monkeypatch, latent, how):
    from latentq_llm_amd import quant as Q
    shapes = [(256, 512), (256, 256), (128, 640)]
    plain = Q.MyAdam.update_step
    seen = []

    def watching(self, group, p, gindex, pindex):
        plain(self, group, p, gindex, pindex)
        seen.append(_seen(self, p))

    a, b = _weights(latent, shapes), _weights(latent, shapes)
    if how == "subclass":
        opt = _adam(a, type("Watching", (Q.MyAdam,), {"update_step": watching}))
    else:
        opt = _adam(a)
    ref = _adam(b)
    if how == "instance":
        opt.update_step = watching.__get__(opt)
    for step in range(3):
        _grads(a, step)
        _grads(b, step)
        if how == "class":
            with monkeypatch.context() as m:
                m.setattr(Q.MyAdam, "update_step", watching)
                opt.step()
        else:
            opt.step()
        ref.step()
        assert len(seen) == len(a)
        for got, w in zip(seen, b):
            for x, y in zip(got, _seen(ref, w)):
                assert torch.equal(x, y) if torch.is_tensor(y) else x is y
        seen.clear()


@pytest.mark.parametrize("latent", ["sr", "w4", "w8"])
def test_a_failing_launch_leaves_codes_and_gradients(hip_lib, monkeypatch, latent):
    from latentq_llm_amd import ops
    weights = _weights(latent, [(256, 512), (256, 256)])
    opt = _adam(weights)
    for step in range(2):  # the first step of a residual goes through the chain
        _grads(weights, step)
        opt.step()
    _grads(weights, 2)
    before = [(w.data, w.data.clone(), w.grad, getattr(w.residual, "lock_mu", None)) for w in weights]
    with monkeypatch.context() as m:
        def fail(queue):
            raise RuntimeError("no launch")
        m.setattr(ops, "adam8_run", fail)
        with pytest.raises(RuntimeError, match="no launch"):
            opt.step()
    for w, (data, codes, grad, mu) in zip(weights, before):
        assert w.data is data and torch.equal(w.data, codes) and w.grad is grad and getattr(w.residual, "lock_mu", None) == mu
    assert opt._queue is None and not opt._in_step


def test_waiting_steps_keep_little_memory(hip_lib):
    """Twelve 4096 x 2048 weights with int8 gradients: a bf16 copy of a gradient is 16 MiB, new codes 4 MiB. 64 MiB may wait,
    one parameter beyond that, and what a parameter's step takes by itself."""
    from latentq_llm_amd import quant as Q
    weights = _weights("sr", [(4096, 2048)] * 12, gbit=8)
    opt = _adam(weights)
    peaks = []
    for step in range(2):
        for w in weights:
            if not isinstance(w.grad, Q.GradientQTensor):
                w.grad = Q.GradientQTensor(list(w.shape), bit=8)
            w.grad.set_value((torch.randn(tuple(w.shape), device="cuda") * 1e-2).to(torch.bfloat16))
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        opt.step()
        peaks.append(torch.cuda.max_memory_allocated() - base)
    assert peaks[1] < (64 + 20 + 20) << 20, peaks


def test_a_parameter_listed_twice_takes_one_step(hip_lib):
    w, = _weights("sr", [(256, 512)])
    v, = _weights("sr", [(256, 512)])
    opt, ref = _adam([w, w]), _adam([v])
    for step in range(2):
        _grads([w], step)
        _grads([v], step)
        opt.step()
        ref.step()
        assert opt.state[w]["step"] == step + 1 and torch.equal(w.data, v.data)
