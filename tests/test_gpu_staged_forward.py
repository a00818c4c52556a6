"""The A16W4 forward for few workgroups (row tiles of 32, 64 and 128 tokens, K cut into slices of 128-k groups): token
counts around the tile heights, a last tile of 16 columns, odd group counts, an uneven last slice, with and without a
split workspace."""
import pytest
import torch

from tests.util import make_w4

pytestmark = pytest.mark.gpu

# one rounding to bf16: at most 2^-9 of an element, so 2^-9 of the norm of the product; as much again for the order of
# the fp32 sums and the rounding of a bias
TOL = 2.0 ** -8


@pytest.fixture(scope="module")
def ops(hip_lib):
    from latentq_llm_amd import ops as o
    return o


@pytest.mark.parametrize("M,N,K", [(18, 4112, 4224), (31, 2032, 11648), (32, 8208, 4096), (33, 4112, 128), (33, 16, 9344), (65, 16, 640), (64, 4112, 1152),
                                   (65, 4112, 1664), (96, 528, 256), (127, 5504, 2048), (128, 2048, 5504), (129, 1040, 1408),
                                   (257, 4112, 384), (385, 2048, 2048), (513, 2064, 8320), (700, 4096, 8192), (1000, 4096, 1152)])
def test_staged_forward(ops, M, N, K):
    kernel, _, _ = ops.a16w4_plan(M, (N, K))
    assert kernel == "staged_128x128"
    _, packed, scales, zeros = make_w4(N, K, M + N + K)
    w = (packed.cuda(), scales.cuda(), zeros.cuda())
    W = ops.a16w4_dequant(*w, (N, K)).float()
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    b = torch.randn(N, device="cuda", generator=g).to(torch.bfloat16)
    ref = x.float() @ W.t()
    for bias in (None, b):
        want = ref if bias is None else ref + b.float()
        y = ops.a16w4_forward(x, *w, (N, K), bias=bias).float()
        assert ((y - want).norm() / want.norm()).item() < TOL
    # rows that pick one k each: exactly the dequantised weights, whichever tile and slice they fall into
    pick = torch.arange(M, device="cuda") * 37 % K
    eye = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16)
    eye[torch.arange(M, device="cuda"), pick] = 1.0
    assert torch.equal(ops.a16w4_forward(eye, *w, (N, K)).float(), W[:, pick].t())
