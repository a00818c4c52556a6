"""The optimizer step whose direction goes straight into the stochastic-rounding requantizer: equal bit for bit to the
two separate calls, at block counts that leave workgroups partly empty, for both block sizes, on groups outside the
requantizer's one-fma form and on operands outside the short square-root and division sequences."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _state(n, block, gen, dev):
    nblk = n // block
    def u8():
        return torch.randint(0, 256, (n,), generator=gen, dtype=torch.uint8).to(dev)
    def f32(scale):
        return (torch.rand(nblk, 1, generator=gen) * scale + scale * 1e-3).to(dev)
    # (codes, scale, max) of each moment; the second holds sqrt(v) + eps: max >= 255 * scale
    s1, s2 = f32(1e-5), f32(1e-5)
    return [u8(), s1, s1 * 128, u8(), s2, s2 * 256]


@pytest.mark.parametrize("N,K,block", [(16, 128, 2048), (48, 128, 2048), (1, 128, 128), (17, 128, 128), (63, 384, 128),
                                       (96, 512, 2048)])
def test_sr_step_equals_adam_then_requant(hip_lib, N, K, block):
    from latentq_llm_amd import ops
    from tests.util import make_w4
    dev, n = torch.device("cuda:0"), N * K
    gen = torch.Generator().manual_seed(N + K)
    _, packed, scales, zeros = make_w4(N, K, 3)
    zeros[::5] += 0.5           # not an integer: no one-fma dequantisation
    scales[1::7] = 2.0 ** -110  # outside its range
    codes, scales, zeros = packed.to(dev), scales.to(dev), zeros.to(dev)
    a = _state(n, block, gen, dev)
    b = [t.clone() for t in a]
    for step in range(3):
        grad = (torch.randn(N, K, generator=gen) * 1e-3).to(torch.bfloat16)
        if step == 1:
            grad[:, ::3] = 0            # zeros
            grad[:, 1::16] = 1e-38      # second moments below 2^-100 where the old ones are tiny
            grad[0, :8] = 1e30          # quotients and squares out of range
        grad = grad.to(dev)
        direction = torch.empty_like(grad)
        ops.adam8_update(grad, a[0], a[3], a[1], a[2], a[4], a[5], 0.9, 0.95, 1e-8, 2e-3, direction=direction)
        want = ops.requant_sr(codes, scales, zeros, direction, 2e-3, (N, K), seed=11, offset=5 + step)
        got = ops.adam8_update(grad, b[0], b[3], b[1], b[2], b[4], b[5], 0.9, 0.95, 1e-8, 2e-3,
                               requant=(codes, scales, zeros, (N, K), 11, 5 + step))
        assert torch.equal(got, want)
        for x, y in zip(a, b):
            assert torch.equal(x.view(torch.uint8) if x.dtype == torch.uint8 else x.view(torch.int32),
                               y.view(torch.uint8) if y.dtype == torch.uint8 else y.view(torch.int32))
        codes = got


@pytest.mark.parametrize("block", [2048, 128])
def test_step_on_operands_outside_the_short_sequences(hip_lib, block):
    """Zero and tiny moments, zero gradients, huge gradients: the parameter, the direction and the moments equal the
    chain of tensor operations bit for bit."""
    from latentq_llm_amd import ops
    from latentq_llm_amd import quant as Q
    dev, n = torch.device("cuda:0"), 2048 * 3
    gen = torch.Generator().manual_seed(block)
    nblk = n // block
    st = [torch.zeros(n, dtype=torch.uint8, device=dev), torch.full((nblk, 1), 1e-10, device=dev), torch.zeros(nblk, 1, device=dev),
          torch.zeros(n, dtype=torch.uint8, device=dev), torch.full((nblk, 1), 1e-10, device=dev), torch.zeros(nblk, 1, device=dev)]
    p = (torch.randn(n, generator=gen) * 0.02).to(torch.bfloat16).to(dev)
    for step in range(3):
        grad = (torch.randn(n, generator=gen) * 1e-3).to(torch.bfloat16)
        grad[::3] = 0
        grad[1::16] = 1e-30
        grad[5:9] = 1e18
        grad = grad.to(dev)
        m = Q.DeQfunc_8bit_opt(st[0], [st[1], st[2]]).to(torch.bfloat16)
        s2 = Q.DeQfunc_8bit_opt(st[3], [st[4], st[5]])
        v = (s2 * s2).to(torch.bfloat16)
        m.mul_(0.9).add_(grad, alpha=1 - 0.9)
        v.mul_(0.95).addcmul_(grad, grad, value=1 - 0.95)
        d = v.sqrt_().add_(1e-8)
        want_p = p.clone().addcdiv_(m, d, value=-1e-3)
        want_dir = m / d
        q1, (w1, h1) = Q.Qfunc_8bit_opt(m.float(), blocksize=nblk)
        q2, (w2, h2) = Q.Qfunc_8bit_opt(d.float(), blocksize=nblk)
        other = [t.clone() for t in st]
        direction = torch.empty_like(grad)
        ops.adam8_update(grad, other[0], other[3], other[1], other[2], other[4], other[5], 0.9, 0.95, 1e-8, 1e-3, direction=direction)
        ops.adam8_update(grad, st[0], st[3], st[1], st[2], st[4], st[5], 0.9, 0.95, 1e-8, 1e-3, param=p)
        assert torch.equal(p, want_p) and torch.equal(direction, want_dir)
        for x, y, w in zip(st, other, (q1, w1, h1, q2, w2, h2)):
            assert torch.equal(x, w) and torch.equal(y, w)


@pytest.mark.parametrize("wbit,lr", [(4, 2e-5), (4, 1e-3), (8, 2e-6)])
def test_step_that_chooses_the_residual_curve_fused_equals_the_chain(hip_lib, monkeypatch, wbit, lr):
    """Every mu_updata_f steps after step 250 the residual codec's curve is chosen from the step itself: chosen curve,
    codes, residual words and moments equal the chain of tensor operations, and the fused kernels ran."""
    from latentq_llm_amd import ops
    from latentq_llm_amd import quant as Q
    from tests.util import make_w4
    N, K = 256, 512

    def run(fused):
        monkeypatch.setattr(Q, "FUSED_ADAM8", fused)
        g = torch.Generator().manual_seed(4)
        weights = []
        for i in range(2):
            if wbit == 4:
                layer = Q.QLinearA16W4(K, N, bias=False, lbit=4, gbit=16)
                _, packed, s, z = make_w4(N, K, 5 + i)
                layer.scales.data, layer.zeros.data = s.cuda(), z.cuda()
                layer.weight.set_value(packed.cuda(), [layer.scales, layer.zeros, layer.wshape])
            else:
                layer = Q.QLinearA8W8(K, N, bias=False, lbit=4, gbit=16)
                layer.qscales.data = ((torch.randn(N, 1, generator=g) * 3e-4).abs() + 1e-5).to(torch.bfloat16).cuda()
                layer.weight.set_value(torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda(), layer.qscales)
            weights.append(layer.weight)
        opt = Q.MyAdam([{"params": weights}], lr=lr, betas=(0.9, 0.95), obit=8, mu_updata_f=20)
        torch.manual_seed(9)
        for step in range(5):
            for w in weights:
                w.grad = (torch.randn(N, K, generator=g) * 1e-3).to(torch.bfloat16).cuda()
                if step == 2:
                    opt.state[w]["step"] = 257  # the next but one step is number 259
            opt.step()
        out = []
        for w in weights:
            s = opt.state[w]
            assert s["step"] == 260
            out += [torch.tensor(w.residual.mu), torch.tensor(w.residual.lock_mu), w.data, w.residual.residual_int] + [
                s[k] for k in ("state1", "qmap1", "absmax1", "state2", "qmap2", "absmax2")]
        return out

    calls = []
    real = ops.adam8_ratio
    monkeypatch.setattr(ops, "adam8_ratio", lambda *a: (calls.append(1), real(*a))[1])
    fused = run(True)
    assert len(calls) == 2
    plain = run(False)
    assert len(calls) == 2
    for x, y in zip(fused, plain):
        assert torch.equal(x.cpu(), y.cpu())
    if lr < 1e-4:
        assert int(fused[0]) == 2  # the curve did change


@pytest.mark.parametrize("block", [2048, 128])
def test_subnormal_second_moments_without_eps(hip_lib, block):
    """The block's minimum is that of its elements where the hardware's square root takes a subnormal for zero. Between these
    two gradients the new scale's last place tells the smaller root (2^-64.5) from zero."""
    from latentq_llm_amd import ops
    from latentq_llm_amd import quant as Q
    from tests.test_gpu_adam8 import chain_step, fresh_state
    n = 4096
    state = fresh_state(n, n // block, torch.device("cuda"))
    fused = {k: t.clone() for k, t in state.items()}
    grad = torch.full((n,), 2.0 ** -64.5, dtype=torch.bfloat16, device="cuda")
    grad[::64] = 8.8470897e-16
    want, step_size = chain_step(Q, grad, state, 1, 1e-3, (0.9, 0.0), 0.0)
    got = torch.empty_like(grad)
    ops.adam8_update(grad, fused["state1"], fused["state2"], fused["qmap1"], fused["absmax1"], fused["qmap2"], fused["absmax2"],
                     0.9, 0.0, 0.0, step_size, direction=got)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    for k, t in state.items():
        assert torch.equal(fused[k].view(-1), t.view(-1)), k
