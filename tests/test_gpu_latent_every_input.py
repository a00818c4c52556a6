"""The latent re-quantisers on all 65 536 bf16 patterns (halves of every size, both clamps, carries, infinities), for scales on both
sides of the reciprocal's range and zero points with and without a fraction, against the chain of tensor operations."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CURVES = [(2, 0.125, 4, 0.25), (2, 0.2666300266320331, 4, 0.375), (2, 0.4330623539159437, 4, 0.46875)]
EVERY = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)


def finite_words(latent):
    return ~torch.isnan(latent.float()).view(-1, 8).any(dim=1)


@pytest.mark.parametrize("curve", CURVES)
@pytest.mark.parametrize("scale,zero", [(1.0, 0.0), (1.0, 8.0), (0.0123, 7.0), (3.0, 7.5), (2.0 ** -50, 8.0)])
def test_w4(hip_lib, curve, scale, zero):
    from latentq_llm_amd import ops
    from oracle import torch_ref as tr
    p1, y1, p2, y2 = curve
    N, K = 512, 128
    latent = EVERY.view(N, K)
    s, z = (torch.full((N, 1), v, dtype=torch.bfloat16) for v in (scale, zero))
    want_codes, want_res = tr.latent_w4_requant(latent.clone(), s, z, (N, K), curve)
    res = torch.empty(N * K // 8, dtype=torch.int32, device="cuda")
    got = ops.latent_w4_requant(latent.cuda(), s.cuda(), z.cuda(), res, (N, K), p1, y1, p2 - p1, y2, 8 - p2)
    words = finite_words(latent)
    assert torch.equal(got.cpu().view(torch.int32)[words], want_codes.contiguous().view(torch.int32)[words])
    assert torch.equal(res.cpu()[words], want_res[words])
    assert int(got.cpu().view(torch.int32)[torch.isnan(latent.float()).view(-1, 8).all(dim=1)].abs().sum()) == 0  # NaN: code 0


@pytest.mark.parametrize("curve", CURVES)
@pytest.mark.parametrize("scale", [1.0, 0.0123, 2.0 ** -50])
def test_w8(hip_lib, curve, scale):
    from latentq_llm_amd import ops
    from oracle import torch_ref as tr
    p1, y1, p2, y2 = curve
    N, K = 512, 128
    latent = EVERY.view(N, K)
    s = torch.full((N, 1), scale, dtype=torch.bfloat16)
    want_codes, want_res = tr.latent_w8_requant(latent.clone(), s, curve)
    res = torch.empty(N * K // 8, dtype=torch.int32, device="cuda")
    got = ops.latent_w8_requant(latent.cuda(), s.cuda(), res, p1, y1, p2 - p1, y2, 8 - p2)
    words = finite_words(latent)
    keep = ~torch.isnan(latent.float())
    assert torch.equal(got.cpu()[keep], want_codes[keep]) and int(got.cpu()[~keep].abs().sum()) == 0
    assert torch.equal(res.cpu()[words], want_res[words])
