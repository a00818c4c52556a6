"""The A16W4 forward in 128-row tiles, on four waves and on eight: both sides of the line for pieces of codes in one cache line and
across two (rows of an odd number of groups, slices that begin at an odd one), each remainder of the loop over three stages, a
single group, whole and cut reductions, an uneven last slice, ragged rows and columns, scales and zeros that are only 2-byte
aligned."""
import pytest
import torch

from tests.util import make_w4

pytestmark = pytest.mark.gpu

# one rounding to bf16: at most 2^-9 of an element, so 2^-9 of the norm of the product; as much again for the order of the fp32
# sums and the rounding of a bias
TOL = 2.0 ** -8


@pytest.mark.parametrize("M,N,groups,slices", [(336, 7808, 11, 1), (1100, 2064, 3, 1), (1100, 2064, 1, 1), (1100, 2064, 31, 1), (379, 3840, 73, 2),
                                               (245, 3072, 57, 5), (800, 2816, 66, 1), (245, 4096, 68, 4), (245, 4096, 76, 4), (380, 4608, 46, 2),
                                               (380, 4608, 54, 2), (500, 2944, 62, 2), (500, 2944, 66, 2), (300, 4096, 116, 2), (300, 4096, 120, 2)])
def test_forward(hip_lib, M, N, groups, slices):
    from latentq_llm_amd import ops
    K = groups * 128
    assert ops.a16w4_plan(M, (N, K))[:2] == ("staged_128x128", slices)
    _, packed, scales, zeros = make_w4(N, K, M + N + K)
    w = (packed.cuda(), scales.cuda(), zeros.cuda())
    W = ops.a16w4_dequant(*w, (N, K)).double()
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    b = torch.randn(N, device="cuda", generator=g).to(torch.bfloat16)
    ref = x.double() @ W.t()
    shifted = [torch.cat((t[:1], t)).flatten()[1:].view_as(t) for t in w[1:]]
    assert all(t.data_ptr() % 4 for t in shifted)
    for bias in (None, b):
        want = ref if bias is None else ref + b.double()
        y = ops.a16w4_forward(x, *w, (N, K), bias=bias)
        assert ((y.double() - want).norm() / want.norm()).item() < TOL
        assert torch.equal(y, ops.a16w4_forward(x, w[0], *shifted, (N, K), bias=bias))
    # rows that pick one k each: exactly the dequantised weights, whichever tile and slice they fall into
    pick = torch.arange(M, device="cuda") * 37 % K
    eye = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16)
    eye[torch.arange(M, device="cuda"), pick] = 1.0
    assert torch.equal(ops.a16w4_forward(eye, *w, (N, K)).double(), W[:, pick].t())
