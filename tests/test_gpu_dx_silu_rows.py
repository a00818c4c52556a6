"""The gradient product with the SiLU backward in its epilogue: a row's result does not depend on how many rows there are."""
import pytest
import torch

from tests.util import make_w4, randn_bf16

pytestmark = pytest.mark.gpu


# one row, edges of the 32 rows that an epilogue asks for at once, of a wave's 64 and of both tile heights
@pytest.mark.parametrize("M", [1, 31, 33, 64, 127, 129, 255, 257, 1025])
def test_rows(M):
    from latentq_llm_amd import ops
    full, N, K = 2100, 320, 1408
    _, packed, scales, zeros = make_w4(N, K, 3)
    w = (packed.cuda(), scales.cuda(), zeros.cuda())
    dy, g, u = randn_bf16((full, N), 4).cuda(), randn_bf16((full, K), 6, 2.0).cuda(), randn_bf16((full, K), 7).cuda()
    want = ops.a16w4_dx_silu_bwd(dy, *w, (N, K), g, u)
    last = full - M  # the last rows, so that a read past the end of M would meet other rows in front
    for rows in (slice(0, M), slice(last, full)):
        got = ops.a16w4_dx_silu_bwd(dy[rows].contiguous(), *w, (N, K), g[rows].contiguous(), u[rows].contiguous())
        for a, b in zip(got, want):
            assert torch.equal(a, b[rows])
