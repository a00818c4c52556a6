"""Input gradients on tiles of 192 rows, whole and in slices: a last tile of one row and a full one, slices that end inside a product
of two, int8 weights, the SiLU backward. A tile's height changes no bit: a few of the tokens alone, which take other heights, have
the same rows."""
import pytest
import torch

from tests.util import make_w4, randn_bf16

pytestmark = pytest.mark.gpu
EPS32, EPS16 = 2.0 ** -24, 2.0 ** -8  # half a unit in the last place of 24 and of 8 significant bits, relative to 1.0


def weights(N, K, seed):
    from latentq_llm_amd import ops
    _, p, s, z = make_w4(N, K, seed)
    w = (p.cuda(), s.cuda(), z.cuda())
    return w, ops.a16w4_dequant(*w, (N, K)).double()


def check(got, pairs):
    """bf16 of an fp32 sum of products in any order: n eps of the sum of magnitudes and one rounding"""
    want, size = sum(d.double() @ w for d, w in pairs), sum(d.double().abs() @ w.abs() for d, w in pairs)
    n = sum(d.shape[1] for d, _ in pairs)
    assert bool(((got.double() - want).abs() <= want.abs() * EPS16 + size * (n + 8) * EPS32).all())


@pytest.mark.parametrize("M,N,K", [(576, 128, 6656), (577, 512, 6656), (700, 512, 5504), (1153, 512, 3328), (1345, 512, 3072)])
def test_whole(hip_lib, M, N, K):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K), backward=True, compute_units=256) == ("staged_192x128", 1, 0)
    (w, W), dy = weights(N, K, 3), randn_bf16((M, N), M).cuda()
    dx = ops.a16w4_dx(dy, *w, (N, K))
    check(dx, [(dy, W)])
    for rows in (slice(0, 130), slice(M - 65, M)):
        few = dy[rows].contiguous()
        if ops.a16w4_plan(few.shape[0], (N, K), backward=True)[1] == 1:
            assert torch.equal(ops.a16w4_dx(few, *w, (N, K)), dx[rows])
    base = randn_bf16((M, K), 5).cuda()
    acc = base.clone()
    ops.a16w4_dx(dy, *w, (N, K), out=acc, accumulate=True)
    assert torch.equal(acc, base + dx)


@pytest.mark.parametrize("M,N,K", [(129, 2048, 5504), (191, 3072, 5504), (257, 3072, 3712), (577, 3072, 3328)])
def test_slices(hip_lib, M, N, K):
    from latentq_llm_amd import ops
    kernel, slices, _ = ops.a16w4_plan(M, (N, K), backward=True, compute_units=256)
    assert kernel == "staged_192x128" and slices > 1
    (w, W), dy = weights(N, K, 3), randn_bf16((M, N), M).cuda()
    check(ops.a16w4_dx(dy, *w, (N, K)), [(dy, W)])
    # a pair of half as many rows each is planned as the one product
    ws, dys = [weights(N // 2, K, seed) for seed in (1, 2)], [randn_bf16((M, N // 2), seed).cuda() for seed in (3, 4)]
    check(ops.a16w4_dx_pair(dys[0], ws[0][0], dys[1], ws[1][0], (N // 2, K), split=True), [(d, w[1]) for d, w in zip(dys, ws)])
    gen = torch.Generator(device="cuda").manual_seed(M)
    w8 = torch.randint(-128, 128, (N, K), generator=gen, device="cuda", dtype=torch.int8)
    qs = (torch.rand(N, generator=gen, device="cuda") * 0.01 + 1e-3).to(torch.bfloat16)
    check(ops.a8w8_dx(dy, w8, qs), [(dy, (w8.to(torch.bfloat16) * qs[:, None]).to(torch.bfloat16).double())])


@pytest.mark.parametrize("M,N,K,rows", [(716, 2048, 6400, 192), (769, 2048, 6400, 192), (577, 128, 6656, 128)])
def test_silu_backward(hip_lib, M, N, K, rows):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K), silu=True, compute_units=256) == ("staged_%dx128" % rows, 1, 0)
    w, _ = weights(N, K, 3)
    dy, g, u = randn_bf16((M, N), 4).cuda(), randn_bf16((M, K), 6, 2.0).cuda(), randn_bf16((M, K), 7).cuda()
    want = ops.a16w4_dx_silu_bwd(dy, *w, (N, K), g, u)
    for rows in (slice(0, 130), slice(M - 65, M)):
        for a, b in zip(ops.a16w4_dx_silu_bwd(dy[rows].contiguous(), *w, (N, K), g[rows].contiguous(), u[rows].contiguous()), want):
            assert torch.equal(a, b[rows])
