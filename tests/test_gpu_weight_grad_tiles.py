"""The three forms of the weight-gradient GEMM choose their tiles by themselves, so that a store of 256 x 256 tiles can meet
accumulating forms of 128 x 128 ones: the tokens fall into the same slices for all of them, and the forms agree in every
bit for any number of tokens."""
import pytest
import torch

from tests.util import randn_bf16, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(hip_lib):
    from latentq_llm_amd import ops
    return ops


FORMS = ("store", "add", "int8")
SMALL, MEDIUM, LARGE, LONE = (128, 128, 4), (192, 256, 8), (256, 256, 8), (256, 256, 4)
# tiles of (store, add, int8), on 256 compute units; a short first step of less and of more than half of a large tile's, rows and columns
# beyond the last whole tile
MIXED = [(121, 2096, 3744, (SMALL, MEDIUM, SMALL)), (33, 2112, 3824, (SMALL, MEDIUM, SMALL)), (59, 3080, 5136, (MEDIUM, SMALL, SMALL)),
         (116, 4784, 3344, (MEDIUM, SMALL, SMALL)), (54, 3672, 3184, (LARGE, LARGE, SMALL)), (97, 2352, 4960, (LARGE, LARGE, SMALL)),
         (461, 4528, 2576, (LARGE, LARGE, SMALL)), (1537, 10760, 4096, (LONE, LONE, SMALL)), (1601, 3336, 3600, (LONE, LONE, LARGE))]


@pytest.mark.parametrize("M,N,K,tiles", MIXED)
def test_tiles_differ(ops, M, N, K, tiles):
    assert tuple(ops.weight_grad_plan(form, M, (N, K), 256) for form in FORMS) == tiles


# and beside them sizes that all three forms have as 192 x 256 tiles
@pytest.mark.parametrize("M,N,K", [s[:3] for s in MIXED] + [(33, 3072, 3072), (49, 2056, 4112), (97, 3080, 3088), (129, 3072, 3072), (500, 2048, 5504),
                                   (1500, 3072, 3072), (1537, 2048, 5504)])
def test_forms_on_different_tiles_agree(ops, M, N, K):
    dy, x = randn_bf16((M, N), M).cuda(), randn_bf16((M, K), M + 1).cuda()
    dw = ops.weight_grad(dy, x)
    # one bf16 rounding of an fp32 sum: 2^-9 relative, and the sum's own error far below it
    assert rel_l2(dw, dy.double().t() @ x.double()) < 2.5e-3
    g = randn_bf16((N, K), 7).cuda()
    want = g.clone().add_(dw)
    assert torch.equal(ops.weight_grad_acc(dy, x, g), want)
    q, s = torch.empty((N, K), dtype=torch.int8, device="cuda"), torch.empty((N, 1), dtype=torch.bfloat16, device="cuda")
    ops.gradq8_quant(dw, q, s, False, seed=3, offset=0)
    want_q = q.clone()
    ops.gradq8_quant(dw, want_q, s, True, seed=3, offset=99)
    ops.weight_grad_acc8(dy, x, q, s, seed=3, offset=99)
    assert torch.equal(q, want_q)


@pytest.mark.parametrize("N,K,tile", [(3072, 3072, MEDIUM), (3336, 3600, LARGE)])
@pytest.mark.parametrize("M", [33, 47, 48, 63, 81, 112])
def test_short_first_step_of_large_tiles_is_exact(ops, M, N, K, tile):
    """Integers whose sums bf16 holds: every token counts once, in whichever slice of the first step it falls."""
    assert ops.weight_grad_plan("store", M, (N, K), 256) == tile
    gen = torch.Generator().manual_seed(M)
    dy = torch.randint(-1, 2, (M, N), generator=gen).to(torch.bfloat16).cuda()
    x = torch.randint(-1, 2, (M, K), generator=gen).to(torch.bfloat16).cuda()
    want = dy.double().t() @ x.double()  # at most 112 in magnitude
    assert torch.equal(ops.weight_grad(dy, x).double(), want)
