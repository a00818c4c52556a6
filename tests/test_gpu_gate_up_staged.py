"""The gate / up product of 17 tokens and more with a workspace: small row tiles of both matrices and the launch that combines
their partial products, at the edges of the row tiles and of the columns, every tile height cut into slices and whole, and the
weights-direct kernel beyond; against float64 of the matrices rounded to bf16, alone, stored (training form) and into a
caller's buffer."""
import pytest
import torch

from tests.util import make_w4, randn_bf16, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,rows,slices", [(17, 16, 256, 32, 1), (31, 144, 512, 32, 1), (32, 128, 7424, 32, 8), (33, 2048, 768, 32, 1),
                                               (64, 4112, 768, 32, 1), (65, 528, 2048, 32, 4), (127, 256, 4096, 32, 8), (200, 1040, 256, 32, 1),
                                               (257, 64, 2304, 32, 4), (33, 8896, 256, 64, 1), (45, 11008, 768, 64, 1), (49, 1376, 5120, 64, 8),
                                               (71, 8432, 512, 128, 1), (129, 5504, 2048, 128, 1), (66, 2832, 2560, 128, 4), (96, 11008, 512, 0, 0)])
def test_gate_up(M, N, K, rows, slices):
    from latentq_llm_amd import ops
    plan = ops.a16w4_gate_up_plan(M, (N, K))
    assert plan == ("staged_128x128", rows, slices) if rows else plan[0] == "direct_128x256"
    mats, dense = [], []
    for seed in (1, 2):
        _, p, s, z = make_w4(N, K, seed)
        mats.append((p.cuda(), s.cuda(), z.cuda()))
        dense.append(ops.a16w4_dequant(*mats[-1], (N, K)).double())
    x = randn_bf16((M, K), 3).cuda()
    g, u = (x.double() @ w.t() for w in dense)
    want = g * torch.sigmoid(g) * u
    h = ops.a16w4_gate_up_silu(x, *mats, (N, K))
    assert rel_l2(h, want) < 2.5e-3  # one bf16 rounding (2^-9) of fp32 sums
    hs, gs, us = ops.a16w4_gate_up_silu(x, *mats, (N, K), save=True)
    assert torch.equal(hs, h) and rel_l2(gs, g) < 2.5e-3 and rel_l2(us, u) < 2.5e-3
    out = torch.full_like(h, float("nan"))
    assert ops.a16w4_gate_up_silu(x, *mats, (N, K), out=out) is out and torch.equal(out, h)
