"""The stochastic-rounding requantizer on either side of the smallest and largest scales that its short form takes, with updates of some
codes, of many times the range and of none, and negative zeros: against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exponent", [-103, -101, -100, -99, -98, -97, -20, 99, 100, 101])
def test_scales_at_the_line(hip_lib, exponent):
    from latentq_llm_amd import ops
    from oracle import c_oracle as co
    from tests.util import make_w4
    N, K = 24, 256
    _, packed, scales, zeros = make_w4(N, K, exponent + 200)
    gen = torch.Generator().manual_seed(exponent)
    scales = ((1 + torch.rand(scales.shape, generator=gen)) * 2.0 ** exponent).to(torch.bfloat16)
    zeros[1::5], zeros[2::7], zeros[3::11] = -16.0, 240.0, 0.0
    steps = torch.randn(N, K, generator=gen) * 4.0 ** torch.randint(-6, 12, (N, K), generator=gen).float()
    grad = (steps.double() * 2.0 ** exponent).float().to(torch.bfloat16)
    bits = lambda t: t.contiguous().view(torch.int16).numpy().view(np.uint16)
    want = co.requant(packed.numpy(), bits(scales), bits(zeros), bits(grad), 0.5, N, K, seed=5, offset=3)
    got = ops.requant_sr(packed.cuda(), scales.cuda(), zeros.cuda(), grad.cuda(), 0.5, (N, K), seed=5, offset=3)
    assert np.array_equal(got.cpu().numpy().view(np.uint8), want)
