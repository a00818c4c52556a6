"""The forward of 17 to 64 tokens against the weights as they are, (q - z) s in float64 and not rounded to bf16: the GEMV of
fewer tokens keeps to them, and so do the kernels for these sizes. With integer zeros and with zeros that are none, at the edges of the
row tiles, cut into slices and whole, for the kernel of 16 columns per compute unit, the staged kernel and, on very many
columns, the staged kernel with several workgroups per unit."""
import pytest
import torch

from tests.util import make_w4, randn_bf16, rel_l2

pytestmark = pytest.mark.gpu

# What is left is the result's own rounding to bf16: 1.54e-3 of its norm for magnitudes spread evenly over a binade's
# logarithm (2^-8 / sqrt(3), over the root mean square of a number in [1, 2)), 1.64e-3 to 1.67e-3 for the sums here. Rounding the
# weights as well adds 1.47e-3 in squares: 2.21e-3.
TOL = 1.8e-3
FEW, STAGED = "few_x16", "staged_128x128"


@pytest.mark.parametrize("M,N,K,kernel", [(17, 4096, 4096, FEW), (32, 2576, 2560, FEW), (33, 4080, 1664, FEW), (48, 4096, 4096, FEW), (64, 3088, 1024, FEW),
                                          (18, 11008, 4096, STAGED), (32, 4096, 11008, STAGED), (33, 2576, 8192, STAGED), (45, 5504, 2048, STAGED),
                                          (48, 4112, 1152, STAGED), (64, 2048, 7296, STAGED), (33, 2560, 8192, FEW), (48, 1040, 1152, FEW), (64, 2048, 4224, FEW), (31, 20480, 1024, STAGED), (64, 33040, 384, STAGED)])
@pytest.mark.parametrize("zeros", ["integer", "eighths", "large"])
def test_weights_are_not_rounded(M, N, K, kernel, zeros):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K))[0] == kernel
    codes, p, s, z = make_w4(N, K, N + K)
    if zeros == "eighths":
        z += torch.randint(0, 8, z.shape, generator=torch.Generator().manual_seed(K)).to(z.dtype) / 8
    elif zeros == "large":  # beyond the integers of 8 bits, where q - z is no bf16 number; every 50th group
        z[::50] = 300.0
    w = ((codes.cuda().double().view(N, -1, 128) - z.cuda().double().view(N, -1, 1)) * s.cuda().double().view(N, -1, 1)).view(N, K)
    b = randn_bf16((N,), 1).cuda()
    x = randn_bf16((M, K), M).cuda()
    want = x.double() @ w.t()
    ops_w = (p.cuda(), s.cuda(), z.cuda())
    assert rel_l2(ops.a16w4_forward(x, *ops_w, (N, K)), want) < TOL
    assert rel_l2(ops.a16w4_forward(x, *ops_w, (N, K), b), want + b.double()) < TOL


@pytest.mark.parametrize("M,N,K", [(100, 256, 4864), (128, 1024, 1792)])
def test_without_a_workspace(M, N, K):
    """lq_a16w4_fwd, which cannot cut K, ran as GEMV launches up to 128 tokens."""
    from latentq_llm_amd import _C
    codes, p, s, z = (t.cuda() for t in make_w4(N, K, N + K))
    w = ((codes.double().view(N, -1, 128) - z.double().view(N, -1, 1)) * s.double().view(N, -1, 1)).view(N, K)
    x = randn_bf16((M, K), M).cuda()
    y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    _C.call("lq_a16w4_fwd", x.data_ptr(), p.data_ptr(), s.data_ptr(), z.data_ptr(), None, y.data_ptr(), M, N, K, 128,
            torch.cuda.current_stream().cuda_stream)
    assert rel_l2(y, x.double() @ w.t()) < TOL
