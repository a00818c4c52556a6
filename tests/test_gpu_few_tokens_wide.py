"""The forward of 65 to 128 tokens, and of fewer on long rows, in one launch (lq_gemm_few.hip, rows of X in halves of a group): all numbers of token groups, every
form by the length of a row, waves with unequal shares, a last tile of tokens with one row, zeros with a fraction, a bias; the
lines to the staged kernel; infinities and NaN in one token."""
import pytest
import torch

from tests.util import make_w4

pytestmark = pytest.mark.gpu

# against the weights as they are: one rounding to bf16, at most 2^-9 of the norm, and the bias's and the sums' beside it
TOL = 2.0 ** -8

SIZES = [(65, 256, 1024), (80, 1536, 1536), (96, 4096, 4096), (81, 2064, 5376), (90, 3088, 7168), (66, 1024, 3072), (97, 2048, 2048), (113, 512, 1024), (128, 3072, 3072),
         (127, 3088, 3328), (100, 4096, 4096), (112, 4080, 2816), (33, 4096, 4352), (48, 2064, 8064), (49, 3072, 4608), (64, 4080, 7680), (33, 2304, 8448), (48, 4096, 10752),
         (17, 4096, 10752), (80, 1040, 1152), (65, 2064, 1664), (96, 16, 1024), (81, 4080, 6272), (66, 144, 2944), (128, 144, 1920), (100, 2064, 3072), (113, 3088, 3968)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_forward(hip_lib, M, N, K):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K), compute_units=256) == ("few_x16", 1, 0)
    codes, packed, scales, zeros = make_w4(N, K, M + N + K)
    if M % 2:
        zeros = (zeros.float() + 0.375).to(torch.bfloat16)
    w = (packed.cuda(), scales.cuda(), zeros.cuda())
    q = torch.stack((packed.view(torch.uint8) >> 4, packed.view(torch.uint8) & 15), -1).view(N, K // 128, 128).cuda().double()
    W = ((q - w[2].view(N, -1, 1).double()) * w[1].view(N, -1, 1).double()).view(N, K)
    gen = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=gen).to(torch.bfloat16)
    b = torch.randn(N, device="cuda", generator=gen).to(torch.bfloat16)
    ref = x.double() @ W.t()
    for bias, want in ((None, ref), (b, ref + b.double())):
        y = ops.a16w4_forward(x, *w, (N, K), bias=bias).double()
        assert ((y - want).norm() / want.norm()).item() < TOL
    # rows that pick one k each, over all halves, slices and places: the weights rounded once
    dense = ops.a16w4_dequant(*w, (N, K))
    for shift in (0, 5, 11):
        pick = (torch.arange(M, device="cuda") * 131 + shift * 72) % K
        eye = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16)
        eye[torch.arange(M, device="cuda"), pick] = 1.0
        assert torch.equal(ops.a16w4_forward(eye, *w, (N, K)), dense[:, pick].t())
    # one token of an infinity or a NaN: no other row sees it
    clean = ops.a16w4_forward(x, *w, (N, K))
    for value in (float("inf"), float("nan")):
        bad = x.clone()
        bad[7, 300] = value
        y = ops.a16w4_forward(bad, *w, (N, K))
        keep = torch.arange(M, device="cuda") != 7
        assert torch.equal(y[keep], clean[keep]) and not bool(torch.isfinite(y[7]).any())


@pytest.mark.parametrize("M,N,K", [(129, 2048, 2048), (65, 4112, 1024), (97, 2048, 2304), (97, 3072, 3328), (100, 4096, 4352), (65, 3072, 5632), (65, 1024, 3328), (80, 2048, 896),
                                   (80, 1040, 4608), (80, 4096, 7296), (81, 2064, 4736), (97, 1040, 2048), (97, 1024, 2176), (48, 4096, 11008), (49, 4096, 8448), (40, 4080, 8448), (40, 4096, 8320)])
def test_lines(hip_lib, M, N, K):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K), compute_units=256)[0] == "staged_128x128"
