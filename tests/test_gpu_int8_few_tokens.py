"""The int8 product on few tokens (16 columns per workgroup; 64 x 64 tiles) and the one-launch forward that quantises its
activations itself: whole numbers and float32 operations in a fixed order, compared bit for bit."""
import pytest
import torch

from tests.util import randn_bf16

pytestmark = pytest.mark.gpu


def operands(N, K, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w8 = torch.randint(-128, 128, (N, K), generator=gen, device="cuda", dtype=torch.int8)
    qs = (torch.rand((N, 1), generator=gen, device="cuda") * 0.01 + 1e-4).to(torch.bfloat16)
    return w8, qs, randn_bf16((N,), seed).cuda()


def product(x8, w8, sx, qs, bias):
    acc = x8.double() @ w8.double().t()
    y = (acc.float() * sx[:, None]) * qs.float().view(1, -1)
    return acc, (y if bias is None else y + bias.float()).to(torch.bfloat16)


# 1, 16, 17 and 32 tokens (one and two groups), 33 (tiles), 64 / 65 rows of a tile; 1, 8, 9 and 33 units of 128 k
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (16, 48, 1024), (17, 2048, 1152), (32, 80, 4224), (32, 8208, 256), (33, 64, 128),
                                   (64, 2048, 2048), (65, 144, 640), (200, 1040, 896), (512, 2048, 512)])
def test_product(M, N, K):
    from latentq_llm_amd import ops
    w8, qs, bias = operands(N, K, M + N)
    x8 = torch.randint(-128, 128, (M, K), device="cuda", dtype=torch.int8, generator=torch.Generator(device="cuda").manual_seed(M))
    sx = torch.rand(M, device="cuda") + 1e-3
    for b, sw in ((bias, qs), (None, qs.float().view(-1))):
        acc, want = product(x8, w8, sx, qs, b)
        y, got_acc = ops.a8w8_forward(x8, w8, sx, sw, b, want_acc=True)
        assert torch.equal(got_acc.double(), acc) and torch.equal(y, want)
        assert torch.equal(ops.a8w8_forward(x8, w8, sx, sw, b), want)


# the largest token counts and widths the one launch takes, the first it does not, rows no multiple of a thread's share
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (1, 32, 65408), (4, 2048, 2048), (7, 48, 1152), (9, 64, 7168), (16, 64, 3968),
                                   (16, 64, 4096), (17, 64, 256)])
@pytest.mark.parametrize("per_token", [False, True])
@pytest.mark.parametrize("special", ["none", "zero", "negative", "nan", "inf"])
def test_forward_quantises_as_the_separate_passes(M, N, K, per_token, special):
    from latentq_llm_amd import ops
    w8, qs, bias = operands(N, K, M + K)
    x = randn_bf16((M, K), M).cuda()
    if special == "zero":
        x[M // 2] = 0
    elif special == "negative":  # the tensor's clamp value is its maximum, not its largest magnitude
        x = -x.abs() - 0.5
    elif special != "none":
        x[M // 2, K - 3] = float(special)
    if per_token:
        x8, sx = ops.act_quant_i8_per_token(x)
    else:
        x8, sx, _ = ops.act_quant_i8_dynamic(x)
    for b in (bias, None):
        want = ops.a8w8_forward(x8, w8, sx, qs, b)
        assert torch.equal(ops.infer8(x, w8, qs, b, per_token).view(torch.int16), want.view(torch.int16))
        assert torch.equal(ops.infer8(x.view(1, M, K), w8, qs, b, per_token).view(M, N).view(torch.int16), want.view(torch.int16))


# a row of exactly one and two steps of 256 pieces, one piece of 16 beyond, half a step; each number of pieces a thread holds
@pytest.mark.parametrize("M,K", [(3, 2048), (5, 2176), (10, 4096), (12, 4224), (3, 1024), (13, 2560), (5, 8192), (16, 2048)])
def test_rows_in_steps(M, K):
    from latentq_llm_amd import ops
    w8, qs, bias = operands(48, K, M + K)
    x = randn_bf16((M, K), M).cuda()
    for row, at in ((0, K - 1), (M - 1, 0), (M // 2, K // 2)):  # the largest in the last, the first and a middle piece
        x[row, at] = 9.0 + row
    x8, sx = ops.act_quant_i8_per_token(x)
    assert torch.equal(ops.infer8(x, w8, qs, bias, True), ops.a8w8_forward(x8, w8, sx, qs, bias))
