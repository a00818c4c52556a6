"""dX with its reduction cut into slices: the fp32 partial products leave by two ways, by the number of rows."""
import pytest
import torch

from tests.util import make_w4, randn_bf16, rel_l2

pytestmark = pytest.mark.gpu


# both sides of the 192 rows, a last block of 32 rows with one row, blocks of a wave that are all past the end; both tile heights
@pytest.mark.parametrize("M,N,K", [(m, n, k) for m in (32, 191, 192, 193, 225, 256, 257, 500) for n, k in ((2048, 128), (4096, 896))]
                         + [(770, 4096, 2048), (1025, 4096, 2048)])
def test_slices(M, N, K):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K), backward=True)[1] > 1
    _, packed, scales, zeros = make_w4(N, K, 3)
    w = (packed.cuda(), scales.cuda(), zeros.cuda())
    dy = randn_bf16((M, N), M).cuda()
    dx = ops.a16w4_dx(dy, *w, (N, K))
    W = ops.a16w4_dequant(*w, (N, K)).double()
    want = dy.double() @ W
    # half a bf16 ulp of the result (a whole one for what the sums move across a tie), and N additions in fp32
    sums = (dy.double().abs() @ W.abs()) * (N * 2.0 ** -24)
    assert bool(((dx.double() - want).abs() <= want.abs() * 2.0 ** -8 + sums).all())
    assert rel_l2(dx, want) < 2.0 ** -8
