"""The staged forward kernel (lq_gemm_staged.hip) takes groups of 128 k in pairs and scales and zeros in pieces of up to eight:
one group, odd and even numbers of them, slices of K that end in half a pair, pieces cut by the end of a row or of the
matrix, matrices aligned to two bytes only, ragged rows and columns, and the form that writes h itself."""
import pytest
import torch

from tests.util import make_w4

pytestmark = pytest.mark.gpu

# one rounding to bf16: at most 2^-9 of an element, so 2^-9 of the norm of the product; as much again for the order of
# the fp32 sums and the rounding of a bias, and where weights are rounded, 2^-9 more for them
TOL = 1.5 * 2.0 ** -8


def _weights(N, K, seed, offset):
    """codes, scales, zeros on the GPU; offset: scales and zeros begin that many values into a buffer"""
    _, packed, scales, zeros = make_w4(N, K, seed)

    def moved(t):
        buf = torch.zeros(t.numel() + offset, 1, dtype=t.dtype, device="cuda")
        buf[offset:] = t.cuda()
        return buf[offset:]
    return packed.cuda(), moved(scales), moved(zeros)


def _x(M, K):
    return torch.randn(M, K, device="cuda", generator=torch.Generator(device="cuda").manual_seed(M)).to(torch.bfloat16)


SMALL = [(65, 16, 128), (64, 4112, 128), (40, 5504, 256), (64, 4112, 384), (33, 4112, 640), (20, 16400, 1152), (64, 6160, 896),
         (50, 2048, 7552), (128, 144, 3200), (100, 2064, 3456), (300, 528, 1152), (129, 256, 128), (30, 160, 11776), (61, 4112, 3328), (20, 6160, 4352)]
# what the kernels of fewer tokens have of the same kinds
FEW = [(33, 16, 128), (64, 272, 128), (64, 1040, 384), (17, 4112, 640), (20, 8208, 1152), (50, 2048, 5504), (100, 2064, 1408), (30, 160, 11008)]
LARGE = [(500, 1024, 5504), (257, 2048, 11008), (1000, 2064, 8320)]  # (whose alignment the small ones cover)


@pytest.mark.parametrize("M,N,K,offset", [size + (offset,) for offset in (0, 1, 2) for size in SMALL + FEW] + [size + (0,) for size in LARGE])
def test_forward(hip_lib, M, N, K, offset):
    from latentq_llm_amd import ops
    kernel = ops.a16w4_plan(M, (N, K), compute_units=256)[0]
    assert kernel == "staged_128x128" if (M, N, K) in SMALL else (M, N, K) in LARGE or kernel in ("few_x16", "gemv_chunks")
    w = _weights(N, K, M + N + K, offset)
    W = ops.a16w4_dequant(w[0], w[1].clone(), w[2].clone(), (N, K)).double()
    x, b = _x(M, K), _x(1, N)[0]
    ref = x.double() @ W.t()
    for bias, want in ((None, ref), (b, ref + b.double())):
        y = ops.a16w4_forward(x, *w, (N, K), bias=bias).double()
        assert ((y - want).norm() / want.norm()).item() < TOL
    # rows that pick one k each: exactly the dequantised weights, whichever pair, half and slice they fall into
    for shift in (0, 77):
        pick = (torch.arange(M, device="cuda") * 131 + shift * 128) % K
        eye = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16)
        eye[torch.arange(M, device="cuda"), pick] = 1.0
        assert torch.equal(ops.a16w4_forward(eye, *w, (N, K)).double(), W[:, pick].t())


@pytest.mark.parametrize("M,N,K", [(17, 11008, 256), (32, 5520, 768), (45, 11024, 512), (64, 8208, 1280), (100, 5504, 512), (150, 2064, 256),
                                   (40, 144, 7424), (45, 1040, 6912), (55, 5392, 2560), (20, 8176, 2816)])
def test_gate_up(hip_lib, M, N, K):
    from latentq_llm_amd import ops
    mats = [_weights(N, K, s, 0) for s in (1, 2)]
    x = _x(M, K)
    want = [x.double() @ ops.a16w4_dequant(*w, (N, K)).double().t() for w in mats]
    want.insert(0, torch.nn.functional.silu(want[0]) * want[1])
    assert ops.a16w4_gate_up_plan(M, (N, K))[0] == "staged_128x128"
    got = ops.a16w4_gate_up_silu(x, *mats, (N, K), save=True)
    for a, ref in zip(got, want):
        assert ((a.double() - ref).norm() / ref.norm()).item() < TOL
    assert torch.equal(ops.a16w4_gate_up_silu(x, *mats, (N, K)), got[0])
