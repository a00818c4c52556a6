"""Input gradients whose reduction is cut into slices: two products into one output (slices that end in the first product,
span both and lie in the second) and int8 weights. Tile edges: 128 and 256 rows, one and several columns of tiles."""
import pytest
import torch

from tests.util import make_w4, randn_bf16

pytestmark = pytest.mark.gpu
EPS32, EPS16 = 2.0 ** -24, 2.0 ** -8  # half a unit in the last place of 24 and of 8 significant bits, relative to 1.0


def check(got, dys, ws):
    """got = bf16 of an fp32 sum of products: against float64, with the first-order bound of a sum in any order (n eps of
    the sum of magnitudes) plus one bf16 rounding."""
    want = sum(d.double() @ w.double() for d, w in zip(dys, ws))
    size = sum(d.double().abs() @ w.double().abs() for d, w in zip(dys, ws))
    n = sum(d.shape[1] for d in dys)
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * EPS16 + size * (n + 8) * EPS32).all()), float(err.max())


@pytest.mark.parametrize("M,N,K", [(1, 1024, 128), (127, 1088, 256), (128, 1024, 384), (129, 2048, 128), (256, 576, 512),
                                   (257, 1536, 2048), (500, 5504, 2048), (1000, 704, 1024)])
def test_pair_split(M, N, K):
    from latentq_llm_amd import ops
    ws, codes = [], []
    for seed in (1, 2):
        _, p, s, z = make_w4(N, K, seed)
        codes.append((p.cuda(), s.cuda(), z.cuda()))
        ws.append(ops.a16w4_dequant(*codes[-1], (N, K)))
    dys = [randn_bf16((M, N), seed).cuda() for seed in (3, 4)]
    got = ops.a16w4_dx_pair(dys[0], codes[0], dys[1], codes[1], (N, K), split=True)
    check(got, dys, ws)
    # which operands go together: with either gradient zero only the other product is left
    zero = torch.zeros_like(dys[0])
    check(ops.a16w4_dx_pair(dys[0], codes[0], zero, codes[1], (N, K), split=True), dys[:1], ws[:1])
    check(ops.a16w4_dx_pair(zero, codes[0], dys[1], codes[1], (N, K), split=True), dys[1:], ws[1:])


@pytest.mark.parametrize("M,N,K", [(1, 1024, 128), (127, 2112, 256), (129, 2048, 128), (257, 1536, 2048), (2048, 8192, 2048)])
def test_int8_split(M, N, K):
    from latentq_llm_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(M)
    w8 = torch.randint(-128, 128, (N, K), generator=gen, device="cuda", dtype=torch.int8)
    qs = (torch.rand(N, generator=gen, device="cuda") * 0.01 + 1e-3).to(torch.bfloat16)
    dy = randn_bf16((M, N), 5).cuda()
    check(ops.a8w8_dx(dy, w8, qs), [dy], [(w8.to(torch.bfloat16) * qs[:, None]).to(torch.bfloat16)])
