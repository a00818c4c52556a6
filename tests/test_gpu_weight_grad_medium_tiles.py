"""The weight-gradient GEMM's 192 x 256 tiles (on 256 compute units all of SIZES take them in every form): a last tile of 8
rows and of 16 columns, whole ones, first steps of one token to a full one, several rounds, noise given and drawn; every token
counted once, and the three forms the same bits."""
import pytest
import torch

from tests.util import randn_bf16, rel_l2

pytestmark = pytest.mark.gpu

SIZES = [(1, 5504, 2048), (33, 3080, 3088), (64, 3072, 3072), (65, 4616, 2064), (127, 3080, 3088), (129, 5504, 2048), (333, 4616, 2064),
         (1600, 4616, 2320)]
# and beside them, 256 x 256 tiles, and 192 x 256 for the store with 128 x 128 for the two others (117 tokens)
MIXED = [(18, 4488, 2800), (48, 3432, 3632), (117, 2968, 5616), (88, 4328, 2864)]


@pytest.fixture(scope="module")
def ops(hip_lib):
    from latentq_llm_amd import ops
    return ops


@pytest.mark.parametrize("M,N,K", SIZES)
def test_every_token_counts_once(ops, M, N, K):
    """Integers whose sums fp32 holds, and bf16 up to 256; beyond that the one rounding of the exact sum."""
    assert all(ops.weight_grad_plan(form, M, (N, K), 256) == (192, 256, 8) for form in ("store", "add", "int8"))
    gen = torch.Generator().manual_seed(M)
    dy = torch.randint(-1, 2, (M, N), generator=gen).to(torch.bfloat16).cuda()
    x = torch.randint(-1, 2, (M, K), generator=gen).to(torch.bfloat16).cuda()
    assert torch.equal(ops.weight_grad(dy, x), (dy.float().t() @ x.float()).to(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", SIZES + MIXED)
def test_forms_agree(ops, M, N, K):
    dy, x = randn_bf16((M, N), M).cuda(), randn_bf16((M, K), M + 1).cuda()
    dw = ops.weight_grad(dy, x)
    # one bf16 rounding of an fp32 sum: 2^-9 relative, and the sum's own error far below it
    assert rel_l2(dw, dy.double().t() @ x.double()) < 2.5e-3
    g = randn_bf16((N, K), 7).cuda()
    want = g.clone().add_(dw)
    assert torch.equal(ops.weight_grad_acc(dy, x, g), want)
    q, s = torch.empty((N, K), dtype=torch.int8, device="cuda"), torch.empty((N, 1), dtype=torch.bfloat16, device="cuda")
    ops.gradq8_quant(dw, q, s, False, seed=3, offset=0)
    given = (torch.rand((N, K), device="cuda") - 0.5).to(torch.bfloat16)
    for noise in (None, given):
        want_q, got = q.clone(), q.clone()
        ops.gradq8_quant(dw, want_q, s, True, noise=noise, seed=3, offset=99)
        ops.weight_grad_acc8(dy, x, got, s, noise=noise, seed=3, offset=99)
        assert torch.equal(got, want_q)
