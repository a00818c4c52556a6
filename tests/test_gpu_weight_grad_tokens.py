"""The weight-gradient GEMM on any number of tokens: all of its tiles, a short first step of every kind of remainder,
against float64, on integers (exact) and through the two accumulating epilogues."""
import pytest
import torch

from tests.util import randn_bf16, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(hip_lib):
    from latentq_llm_amd import ops
    return ops


# 128 x 128 tiles in steps of 32 tokens, four stages: fewer steps than stages, remainders of 1, 15..17, 31
SMALL = [(1, 64, 128), (15, 136, 72), (31, 128, 128), (32, 128, 136), (33, 256, 264), (65, 128, 384), (96, 200, 128), (113, 128, 128),
         (160, 128, 256), (500, 264, 520)]
# the same tiles on more outputs, and 192 x 256 ones in steps of 64 tokens (97 tokens)
MORE = [(1, 2048, 4096), (40, 2048, 4096), (64, 2048, 4096), (97, 2056, 4104), (193, 2048, 4096)]
# 256 x 256 tiles in steps of 64 tokens, two stages; outputs that end inside a tile
LARGE = [(1, 3336, 3600), (40, 3848, 3856), (64, 4072, 4080), (97, 4104, 3344), (193, 3336, 3600)]


@pytest.mark.parametrize("M,N,K,tile", [s + (None,) for s in SMALL + MORE] + [s + ((256, 256, 8),) for s in LARGE])
def test_weight_grad_any_number_of_tokens(ops, M, N, K, tile):
    if tile:
        assert all(ops.weight_grad_plan(form, M, (N, K), 256) == tile for form in ("store", "add", "int8"))
    dy, x = randn_bf16((M, N), M).cuda(), randn_bf16((M, K), M + 1).cuda()
    dw = ops.weight_grad(dy, x)
    # one bf16 rounding of an fp32 sum: 2^-9 relative, and the sum's own error far below it
    assert rel_l2(dw, dy.double().t() @ x.double()) < 2.5e-3
    g = torch.Generator().manual_seed(M)
    dyi = torch.randint(-1, 2, (M, N), generator=g).to(torch.bfloat16).cuda()
    xi = torch.randint(-1, 2, (M, K), generator=g).to(torch.bfloat16).cuda()
    want = dyi.double().t() @ xi.double()
    assert float(want.abs().max()) <= 256  # integers that bf16 holds
    assert torch.equal(ops.weight_grad(dyi, xi).double(), want)


@pytest.mark.parametrize("M,N,K", [(31, 128, 144), (100, 264, 272), (40, 2048, 4096), (129, 2048, 4096)] + LARGE)
def test_accumulating_epilogues_any_number_of_tokens(ops, M, N, K):
    dy, x = randn_bf16((M, N), 5).cuda(), randn_bf16((M, K), 6).cuda()
    dw = ops.weight_grad(dy, x)
    g = randn_bf16((N, K), 7).cuda()
    want = g.clone().add_(dw)
    assert torch.equal(ops.weight_grad_acc(dy, x, g), want)
    q = torch.empty((N, K), dtype=torch.int8, device="cuda")
    s = torch.empty((N, 1), dtype=torch.bfloat16, device="cuda")
    ops.gradq8_quant(dw, q, s, False, seed=3, offset=0)
    want_q = q.clone()
    ops.gradq8_quant(dw, want_q, s, True, seed=3, offset=99)
    ops.weight_grad_acc8(dy, x, q, s, seed=3, offset=99)
    assert torch.equal(q, want_q)


def test_rows_past_the_last_token_do_not_count(ops):
    """A short first step re-reads its last token row and masks it: an infinity in that row reaches the result once, and
    rows of a larger buffer behind the operands do not reach it at all."""
    M, N, K = 21, 128, 128
    buf_dy, buf_x = torch.full((64, N), float("nan"), dtype=torch.bfloat16), torch.full((64, K), float("nan"), dtype=torch.bfloat16)
    buf_dy[:M], buf_x[:M] = 1.0, 2.0
    dw = ops.weight_grad(buf_dy.cuda()[:M], buf_x.cuda()[:M])
    assert torch.equal(dw, torch.full_like(dw, 42.0))
    buf_dy[M - 1, 3] = float("inf")
    dw = ops.weight_grad(buf_dy.cuda()[:M], buf_x.cuda()[:M])
    assert torch.isinf(dw[3]).all() and torch.equal(dw[4:], torch.full_like(dw[4:], 42.0))


# 1536 tokens and more: on 256 x 256 tiles 4 waves of 128 x 128 where the int8 epilogue has 8 of 128 x 64, or 128 x 128 tiles of its own;
# tokens of every kind of first step, outputs that end inside a tile. And outputs of fewer tiles, which all forms have as 128 x 128
# or 192 x 256 ones.
LONE = (256, 256, 4)


@pytest.mark.parametrize("M,N,K,store,int8", [(1536, 3336, 3600, LONE, (256, 256, 8)), (1537, 10760, 4096, LONE, (128, 128, 4)),
                                              (1586, 3848, 3856, LONE, (256, 256, 8)), (1599, 11000, 4080, LONE, (256, 256, 8)),
                                              (2001, 4104, 3344, LONE, (256, 256, 8)),
                                              (1536, 2048, 4096, (128, 128, 4), (128, 128, 4)), (1537, 2056, 4112, (192, 256, 8), (192, 256, 8)),
                                              (1586, 3080, 3088, (192, 256, 8), (192, 256, 8)), (1599, 4096, 2064, (192, 256, 8), (192, 256, 8))])
def test_four_waves_per_tile(ops, M, N, K, store, int8):
    plans = [ops.weight_grad_plan(form, M, (N, K), 256) for form in ("store", "add", "int8")]
    assert plans == [store, store, int8]
    dy, x = randn_bf16((M, N), M).cuda(), randn_bf16((M, K), M + 1).cuda()
    dw = ops.weight_grad(dy, x)
    assert rel_l2(dw, dy.double().t() @ x.double()) < 2.5e-3  # as above
    gen = torch.Generator().manual_seed(M)
    # few enough terms that every sum is an integer bf16 holds
    dyi = (torch.randint(-1, 2, (M, N), generator=gen) * (torch.rand((M, 1), generator=gen) < 0.1)).to(torch.bfloat16).cuda()
    xi = torch.randint(-1, 2, (M, K), generator=gen).to(torch.bfloat16).cuda()
    want = dyi.double().t() @ xi.double()
    assert float(want.abs().max()) <= 256 and torch.equal(ops.weight_grad(dyi, xi).double(), want)
    g = randn_bf16((N, K), 7).cuda()
    want = g.clone().add_(dw)
    assert torch.equal(ops.weight_grad_acc(dy, x, g), want)
    q, s = torch.empty((N, K), dtype=torch.int8, device="cuda"), torch.empty((N, 1), dtype=torch.bfloat16, device="cuda")
    ops.gradq8_quant(dw, q, s, False, seed=3, offset=0)
    want_q = q.clone()
    ops.gradq8_quant(dw, want_q, s, True, seed=3, offset=99)
    ops.weight_grad_acc8(dy, x, q, s, seed=3, offset=99)
    assert torch.equal(q, want_q)
