"""The forward of 17 to 64 tokens with 16 columns per workgroup: every number of 16-token groups at its edges, K of fewer groups
than waves, of fewer and more than the stages and of every remainder, the first and the last column block."""
import pytest
import torch

from tests.util import make_w4, randn_bf16, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(2064, 128), (4096, 256), (2576, 640), (4080, 1152), (4096, 1664), (3088, 2432), (4096, 4096)])
@pytest.mark.parametrize("bias", [False, True])
def test_forward(N, K, bias):
    from latentq_llm_amd import ops
    _, p, s, z = make_w4(N, K, N + K)
    w = (p.cuda(), s.cuda(), z.cuda())
    dense = ops.a16w4_dequant(*w, (N, K)).double()
    b = randn_bf16((N,), 1).cuda() if bias else None
    for M in (17, 31, 32, 33, 48, 49, 63, 64):
        assert ops.a16w4_plan(M, (N, K))[0] == "few_x16"
        x = randn_bf16((M, K), M).cuda()
        want = x.double() @ dense.t() + (0 if b is None else b.double())
        assert rel_l2(ops.a16w4_forward(x, *w, (N, K), b), want) < 2.5e-3, M  # one bf16 rounding (2^-9) of fp32 sums
    # one token at a time picks one column of the dequantised matrix: exact, so every k reaches its weight
    x = torch.zeros((64, K), dtype=torch.bfloat16, device="cuda")
    k = torch.randperm(K, generator=torch.Generator().manual_seed(K))[:64].cuda()
    x[torch.arange(len(k)), k] = 1.0
    want = dense[:, k].t().to(torch.bfloat16)
    assert torch.equal(ops.a16w4_forward(x, *w, (N, K))[: len(k)], want)
