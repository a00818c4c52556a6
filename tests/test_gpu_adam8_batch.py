"""An optimizer step over many parameters (their fused steps leave together, up to eight to a launch) against the same steps
one parameter at a time: stochastic rounding, int4 and int8 codes with residual, both block sizes, more parameters than a
launch takes, three steps in a row. Bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
# (the smallest keep fp32 moments and take the chain in between)
SHAPES = [(32, 128), (40, 128), (1, 128), (48, 256), (128, 384), (1024, 2048), (33, 128), (81, 128), (64, 512), (3, 128), (256, 256), (65, 128),
          (96, 128)]


def build(seed, copies):
    from latentq_llm_amd import quant as Q
    gen = torch.Generator(device="cuda").manual_seed(seed)
    sets = [[] for _ in range(copies)]
    for i, (n, k) in enumerate(SHAPES * 2):
        groups = n * k // 128
        scales = (torch.rand((groups, 1), generator=gen, device="cuda") * 0.01 + 1e-3).to(torch.bfloat16)
        zeros = torch.randint(6, 10, (groups, 1), generator=gen, device="cuda").to(torch.bfloat16)
        codes = torch.randint(-128, 128, (n * k // 2,), generator=gen, device="cuda", dtype=torch.int8)
        codes8 = torch.randint(-127, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
        qs = (torch.rand((n, 1), generator=gen, device="cuda") * 1e-3 + 1e-4).to(torch.bfloat16)
        for params in sets:
            if i % 3 == 2:
                m = Q.QLinearA8W8(k, n, bias=False, lbit=4, gbit=16)
                m.qscales.data = qs.clone()
                m.weight.set_value(codes8.clone(), m.qscales)
            else:
                m = Q.QLinearA16W4(k, n, bias=False, lbit=0 if i % 3 else 4, gbit=16)
                m.scales.data, m.zeros.data = scales.clone(), zeros.clone()
                m.weight.set_value(codes.clone(), [m.scales, m.zeros, m.wshape])
            params.append(m.weight)
    return sets


def test_a_step_equals_the_steps_of_its_parameters():
    from latentq_llm_amd import quant as Q
    together, alone = build(1, 2)
    make = lambda ws: Q.MyAdam([{"params": ws}], lr=1e-3, betas=(0.9, 0.95), obit=8, sr_seed=5)
    a, b = make(together), make(alone)
    gen = torch.Generator(device="cuda").manual_seed(2)
    for _ in range(3):
        grads = [torch.randn(tuple(w.shape), generator=gen, device="cuda").mul_(1e-2).to(torch.bfloat16) for w in together]
        for w, v, g in zip(together, alone, grads):
            w.grad, v.grad = g.clone(), g.clone()
        a.step()
        for i, v in enumerate(alone):
            if len(b.state[v]) == 0:
                b.init_state(b.param_groups[0], v, 0, i)
            b.update_step(b.param_groups[0], v, 0, i)
        for w, v in zip(together, alone):
            assert w.grad is None and torch.equal(w.data, v.data)
            for k, t in a.state[w].items():
                assert torch.equal(t, b.state[v][k]) if torch.is_tensor(t) else t == b.state[v][k], k
            if w.residual is not None:
                assert torch.equal(w.residual.residual_int, v.residual.residual_int)
    assert a._queue is None and not a._in_step


def test_a_failing_parameter_leaves_the_others_updated():
    from latentq_llm_amd import quant as Q
    together, alone = build(3, 2)
    a = Q.MyAdam([{"params": together[:4]}], lr=1e-3, betas=(0.9, 0.95), obit=8)
    b = Q.MyAdam([{"params": alone[:3]}], lr=1e-3, betas=(0.9, 0.95), obit=8)
    for w, v in zip(together[:4], alone[:4]):
        w.grad = torch.full(tuple(w.shape), 1e-2, dtype=torch.bfloat16, device="cuda")
        v.grad = w.grad.clone()
    plain = a.update_step

    def update(group, p, gindex, pindex):
        if pindex == 3:
            raise RuntimeError("stop")
        plain(group, p, gindex, pindex)

    a.update_step = update
    with pytest.raises(RuntimeError, match="stop"):
        a.step()
    b.step()
    for w, v in zip(together[:3], alone[:3]):
        assert torch.equal(w.data, v.data)
