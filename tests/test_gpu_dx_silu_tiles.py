"""The gradient product with the SiLU backward in its epilogue, on both tile heights: which one runs follows from the sizes, and a
row has the same result on either."""
import pytest
import torch

from tests.util import make_w4, randn_bf16

pytestmark = pytest.mark.gpu


# rows of a tile for all the tokens and for the first of them, on 256 compute units; outputs that end inside a tile
@pytest.mark.parametrize("full,few,N,K,heights", [(1928, 257, 2560, 7936, (256, 128)), (1916, 130, 3584, 8064, (256, 128)),
                                                  (716, 257, 2048, 6400, (192, 128)), (1928, 716, 2048, 6400, (256, 192))])
def test_tile_heights_agree(full, few, N, K, heights):
    from latentq_llm_amd import ops
    for M, rows in zip((full, few), heights):
        assert ops.a16w4_plan(M, (N, K), silu=True, compute_units=256) == ("staged_%dx128" % rows, 1, 0)
    _, packed, scales, zeros = make_w4(N, K, 3)
    w = (packed.cuda(), scales.cuda(), zeros.cuda())
    dy, g, u = randn_bf16((full, N), 4).cuda(), randn_bf16((full, K), 6, 2.0).cuda(), randn_bf16((full, K), 7).cuda()
    want = ops.a16w4_dx_silu_bwd(dy, *w, (N, K), g, u)
    for rows in (slice(0, few), slice(full - few, full)):
        got = ops.a16w4_dx_silu_bwd(dy[rows].contiguous(), *w, (N, K), g[rows].contiguous(), u[rows].contiguous())
        for a, b in zip(got, want):
            assert torch.equal(a, b[rows])
