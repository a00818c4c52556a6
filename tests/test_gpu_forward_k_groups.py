"""The weights-direct forward kernels on grids of at most one workgroup per compute unit, with two groups of waves per workgroup,
each on its part of K, where K is long enough: equal and unequal parts, the shortest K and the one below it, ragged rows and
columns, all tiles."""
import pytest
import torch

from tests.util import make_w4

pytestmark = pytest.mark.gpu

# one rounding to bf16: at most 2^-9 of an element, so 2^-9 of the norm of the product; as much again for the order of
# the fp32 sums and the rounding of a bias
TOL = 2.0 ** -8


@pytest.mark.parametrize("M,N,K,kernel", [(200, 11008, 256, "direct_128x128"), (200, 11008, 512, "direct_128x128"),
                                          (255, 11024, 768, "direct_128x128"), (1000, 4096, 1280, "direct_128x128"),
                                          (513, 4112, 3328, "direct_128x128"), (129, 9008, 7936, "direct_128x128"),
                                          (1900, 4112, 512, "direct_128x256"), (1537, 4096, 1792, "direct_128x256"),
                                          (1000, 4096, 1024, "direct_128x128"), (1000, 4096, 768, "direct_128x128"),
                                          (769, 4112, 8192, "direct_128x128"),
                                          (1900, 4112, 1536, "direct_128x256"), (1900, 4112, 1280, "direct_128x256")])
def test_forward(hip_lib, M, N, K, kernel):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K))[0] == kernel
    _, packed, scales, zeros = make_w4(N, K, M + N + K)
    w = (packed.cuda(), scales.cuda(), zeros.cuda())
    W = ops.a16w4_dequant(*w, (N, K)).double()
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    b = torch.randn(N, device="cuda", generator=g).to(torch.bfloat16)
    ref = x.double() @ W.t()
    for bias, want in ((None, ref), (b, ref + b.double())):
        y = ops.a16w4_forward(x, *w, (N, K), bias=bias).double()
        assert ((y - want).norm() / want.norm()).item() < TOL
    # rows that pick one k each: exactly the dequantised weights, whichever part of K they fall into
    pick = torch.arange(M, device="cuda") * 37 % K
    eye = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16)
    eye[torch.arange(M, device="cuda"), pick] = 1.0
    assert torch.equal(ops.a16w4_forward(eye, *w, (N, K)).double(), W[:, pick].t())


@pytest.mark.parametrize("M,N,K", [(300, 5504, 768), (97, 11024, 512), (257, 5520, 2816), (257, 5520, 3072), (200, 11008, 3328), (513, 6160, 4096), (500, 8192, 3840)])
def test_gate_up(hip_lib, M, N, K):
    from latentq_llm_amd import ops
    mats = [tuple(t.cuda() for t in make_w4(N, K, s)[1:]) for s in (1, 2)]
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    want = [x.double() @ ops.a16w4_dequant(*w, (N, K)).double().t() for w in mats]
    want.insert(0, torch.nn.functional.silu(want[0]) * want[1])
    assert ops.a16w4_gate_up_plan(M, (N, K))[0] == "direct_128x256"
    for got, ref in zip(ops.a16w4_gate_up_silu(x, *mats, (N, K), save=True), want):
        assert ((got.double() - ref).norm() / ref.norm()).item() < TOL
