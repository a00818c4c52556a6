"""The int8 product in 32 x 32 tiles, four waves on a quarter of K each: whole numbers and float32 operations in a fixed order,
compared bit for bit."""
import pytest
import torch

from tests.util import randn_bf16

pytestmark = pytest.mark.gpu


# 33 tokens (the first that tiles take), a tile's last row and the next one's first; 16 columns of a tile; 16 units of 128 k, 17
# and 23 (quarters of unequal length), 64; the largest output of one tile per compute unit, the first beyond, the last short K
@pytest.mark.parametrize("M,N,K", [(33, 16, 2048), (64, 48, 2176), (65, 144, 2944), (128, 2048, 2048), (33, 4096, 2304), (33, 4112, 2304),
                                   (129, 2048, 2048), (256, 1024, 8192), (500, 80, 3072), (40, 2560, 1920)])
def test_product(M, N, K):
    from latentq_llm_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    w8 = torch.randint(-128, 128, (N, K), generator=gen, device="cuda", dtype=torch.int8)
    x8 = torch.randint(-128, 128, (M, K), generator=gen, device="cuda", dtype=torch.int8)
    qs = (torch.rand((N, 1), generator=gen, device="cuda") * 0.01 + 1e-4).to(torch.bfloat16)
    sx = torch.rand(M, generator=gen, device="cuda") + 1e-3
    bias = randn_bf16((N,), M).cuda()
    acc = x8.double() @ w8.double().t()
    for b, sw in ((bias, qs), (None, qs.float().view(-1))):
        y = (acc.float() * sx[:, None]) * qs.float().view(1, -1)
        want = (y if b is None else y + b.float()).to(torch.bfloat16)
        got, got_acc = ops.a8w8_forward(x8, w8, sx, sw, b, want_acc=True)
        assert torch.equal(got_acc.double(), acc) and torch.equal(got, want)
        assert torch.equal(ops.a8w8_forward(x8, w8, sx, sw, b), want)
