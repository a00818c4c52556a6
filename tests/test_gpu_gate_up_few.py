"""The gate / up product of 17 to 64 tokens in one launch (lq_gate_up_few.hip): every number of token groups, one and two blocks of
columns to a workgroup, a last workgroup with one block, shares of K of one to seven groups, even and odd ones; zeros with a
fraction; scales on two bytes only, which other kernels take."""
import pytest
import torch

from tests.util import make_w4, rel_l2

pytestmark = pytest.mark.gpu

SIZES = [(17, 2064, 1024), (32, 4096, 1280), (33, 2080, 7168), (48, 4096, 2304), (49, 4080, 1024), (64, 2064, 5632), (20, 4112, 1024), (31, 7664, 4096),
         (48, 7680, 1280), (45, 5504, 2048), (32, 128, 1280), (33, 2048, 1024), (35, 1376, 3072), (17, 16, 7168), (48, 144, 6656), (64, 1040, 4864)]


def matrices(N, K, offset, frac):
    from latentq_llm_amd import ops
    mats, dense = [], []
    for seed in (1, 2):
        _, p, s, z = make_w4(N, K, seed)
        if frac:
            z = (z.float() + 0.375).to(torch.bfloat16)

        def moved(t):
            buf = torch.zeros(t.numel() + offset, 1, dtype=t.dtype, device="cuda")
            buf[offset:] = t.cuda().view(-1, 1)
            return buf[offset:]
        dense.append(ops.a16w4_dequant(p.cuda(), s.cuda(), z.cuda(), (N, K)).double())
        mats.append((p.cuda(), moved(s), moved(z)))
    return mats, dense


@pytest.mark.parametrize("M,N,K,offset,frac", [s + (0, i % 3 == 2) for i, s in enumerate(SIZES)] + [(17, 2064, 1024, 1, False), (45, 4112, 1280, 1, True)])
def test_gate_up(hip_lib, M, N, K, offset, frac):
    from latentq_llm_amd import ops
    assert ops.a16w4_gate_up_plan(M, (N, K), compute_units=256)[0] == "few_x16"
    assert ops.a16w4_gate_up_plan(M, (N, K), workspace_bytes=0, compute_units=256)[0] == "few_x16"
    mats, dense = matrices(N, K, offset, frac)
    x = torch.randn(M, K, device="cuda", generator=torch.Generator(device="cuda").manual_seed(M)).to(torch.bfloat16)
    g, u = (x.double() @ w.t() for w in dense)
    h = ops.a16w4_gate_up_silu(x, *mats, (N, K))
    assert rel_l2(h, g * torch.sigmoid(g) * u) < 2.5e-3  # one bf16 rounding (2^-9) of fp32 sums
    hs, gs, us = ops.a16w4_gate_up_silu(x, *mats, (N, K), save=True)
    assert torch.equal(hs, h) and rel_l2(gs, g) < 2.5e-3 and rel_l2(us, u) < 2.5e-3
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert ops.a16w4_gate_up_silu(x, *mats, (N, K), out=out) is out and torch.equal(out, h)
    # rows that pick one k each, over the groups and the places in them: the dequantised weights themselves
    for shift in (0, 5, 11):
        pick = (torch.arange(M, device="cuda") * 131 + shift * 128) % K
        eye = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16)
        eye[torch.arange(M, device="cuda"), pick] = 1.0
        _, gs, us = ops.a16w4_gate_up_silu(eye, *mats, (N, K), save=True)
        assert torch.equal(gs.double(), dense[0][:, pick].t()) and torch.equal(us.double(), dense[1][:, pick].t())


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_one_token_of_infinity_or_nan(hip_lib, value):
    """Only its own row, and as the products of the stored weights have it."""
    from latentq_llm_amd import ops
    M, N, K = 40, 4112, 1280
    mats, dense = matrices(N, K, 0, False)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    _, g0, u0 = ops.a16w4_gate_up_silu(x, *mats, (N, K), save=True)
    x[7, 300] = value
    _, g, u = ops.a16w4_gate_up_silu(x, *mats, (N, K), save=True)
    keep = torch.arange(M, device="cuda") != 7
    for got, before, w in ((g, g0, dense[0]), (u, u0, dense[1])):
        assert torch.equal(got[keep], before[keep])
        want = x[7].double()[300] * w[:, 300]
        assert torch.equal(got[7].double().nan_to_num(nan=0.25, posinf=2, neginf=-2), want.nan_to_num(nan=0.25, posinf=2, neginf=-2))
