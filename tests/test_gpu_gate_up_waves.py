"""The gate / up pass of up to 16 tokens: every number of staged rows and of waves its rule picks (one to four workgroups per
compute unit, one to nine batches of 512 k, short last batches, waves without a batch)."""
import pytest
import torch

from tests.util import make_w4, randn_bf16, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(16, 128), (48, 640), (4080, 1536), (4112, 2560), (4128, 3072), (8208, 3584), (8224, 2304),
                                 (8192, 4096), (12304, 1024), (64, 4224), (32, 9216)])
def test_gate_up_few_tokens(N, K):
    from latentq_llm_amd import ops
    mats, dense = [], []
    for seed in (1, 2):
        _, p, s, z = make_w4(N, K, seed)
        mats.append((p.cuda(), s.cuda(), z.cuda()))
        dense.append(ops.a16w4_dequant(*mats[-1], (N, K)).double())
    for M in (1, 4, 5, 8, 9, 12, 13, 16):
        x = randn_bf16((M, K), M).cuda()
        g, u = (x.double() @ w.t() for w in dense)
        want = g * torch.sigmoid(g) * u
        h = ops.a16w4_gate_up_silu(x, *mats, (N, K))
        # the sums are fp32 of exact products, but the pass does not round the weights to bf16 as the dense form does: half
        # a unit in the last place of 8 bits (2^-9 on average over a binade) each on the two products and on the result
        assert rel_l2(h, want) < 5e-3, (M, rel_l2(h, want))
        # a product of every row against the plain pass, which adds the same terms in another order
        y = ops.a16w4_forward(x, *mats[0], (N, K))
        assert rel_l2(y, g) < 5e-3


@pytest.mark.parametrize("N,K", [(4112, 2560), (8208, 3584), (12304, 4096), (16400, 640), (20480, 2048), (8224, 4224), (16400, 8704)])
def test_rows_do_not_depend_on_how_many_there_are(N, K):
    """The launcher picks the waves of a workgroup by the number of rows; the order of the sums stays that of K alone, so 16
    rows have the bits they have among N."""
    from latentq_llm_amd import ops
    mats = []
    for seed in (1, 2):
        _, p, s, z = make_w4(N, K, seed)
        mats.append((p.cuda(), s.cuda(), z.cuda()))
    rows = slice(N - 16, N)
    few = [(p.view(N, -1)[rows].reshape(-1), s.view(N, -1)[rows].reshape(-1, 1), z.view(N, -1)[rows].reshape(-1, 1)) for p, s, z in mats]
    for M in (1, 3, 4, 5, 8, 9, 12, 13, 16):
        x = randn_bf16((M, K), M).cuda()
        assert torch.equal(ops.a16w4_gate_up_silu(x, *mats, (N, K))[:, rows], ops.a16w4_gate_up_silu(x, *few, (16, K))), M


@pytest.mark.parametrize("K", [512 * b - 128 * (b % 3) for b in range(1, 13)] + [8704])
def test_every_form_has_a_kernel(K):
    """One to five workgroups to a unit on one to twelve batches of 512 k, and seventeen: the forms the launcher has to have. Rows
    have the bits they have in the smallest matrix, which the other tests compare with a reference."""
    from latentq_llm_amd import ops
    N = 16400
    mats = []
    for seed in (1, 2):
        _, p, s, z = make_w4(N, K, seed)
        mats.append((p.cuda(), s.cuda(), z.cuda()))
    for M in (4, 8, 12, 16):
        x = randn_bf16((M, K), M).cuda()
        h = {n: ops.a16w4_gate_up_silu(x, *[(p[:n * K // 2], s[:n * K // 128], z[:n * K // 128]) for p, s, z in mats], (n, K))
             for n in (16, 4096, 8192, 12288, 16384, N)}
        for n, y in h.items():
            assert torch.equal(y, h[N][:, :n]) and torch.equal(y[:, :16], h[16]), (M, n)
