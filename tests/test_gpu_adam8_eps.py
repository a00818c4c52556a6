"""The optimizer step where second moments or their roots are tiny, on both sides of the eps from which the kernel does not look
for them: moments from 2^-84 down to zero (through the subnormals), every code of a block, both block sizes, against the tensor
chain, bit for bit."""
import pytest
import torch

from tests.test_gpu_adam8 import chain_step, fresh_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [2048, 128])
@pytest.mark.parametrize("eps", [1e-8, 2.0 ** -38, 2.0 ** -38 * (1 - 2.0 ** -24), 1.2345e-12, 2.0 ** -45, 1e-20, 0.0])
def test_tiny_second_moments(hip_lib, eps, block):
    from latentq_llm_amd import ops, quant as q
    dev, n = torch.device("cuda:0"), 2048 * 6
    g = torch.Generator().manual_seed(3)
    ref = fresh_state(n, n // block, dev)
    fus = {k: v.clone() for k, v in ref.items()}
    for step in range(1, 4):
        grad = torch.randn(n, generator=g) * 2.0 ** torch.randint(-77, -40, (n,), generator=g).float()
        grad[:2048] *= 2.0 ** 40  # a block with ordinary moments, and some nothing in it
        grad[100:110] = 0.0
        grad[5000] = 1e-3         # one ordinary element among tiny ones
        grad = grad.to(torch.bfloat16).to(dev)
        want, step_size = chain_step(q, grad, ref, step, 1e-3, (0.9, 0.95), eps)
        got = torch.empty(n, dtype=torch.bfloat16, device=dev)
        ops.adam8_update(grad, fus["state1"], fus["state2"], fus["qmap1"], fus["absmax1"], fus["qmap2"], fus["absmax2"], 0.9, 0.95, eps,
                         step_size, direction=got)
        for name in ref:
            assert torch.equal(ref[name].view(-1), fus[name].view(-1)), (step, name)
        assert torch.equal(torch.isnan(want), torch.isnan(got))
        assert torch.equal(torch.nan_to_num(want.float()), torch.nan_to_num(got.float())), step
