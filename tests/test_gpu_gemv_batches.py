"""The products of up to 16 tokens by how a wave's batches of four groups of 128 k are loaded: one batch a wave, several with the next
one's codes in flight, several without, two row tiles, and the gate / up pass with one, two and three workgroups to a compute
unit; short last batches, waves without one, every number of staged rows."""
import pytest
import torch

from tests.util import make_w4

pytestmark = pytest.mark.gpu

TOL = 2.0 ** -8  # one rounding to bf16, as much again for the order of the fp32 sums


def _mat(N, K, seed):
    _, packed, scales, zeros = make_w4(N, K, seed)
    w = (packed.cuda(), scales.cuda(), zeros.cuda())
    q = torch.stack([(w[0].view(torch.uint8) >> 4), (w[0].view(torch.uint8) & 15)], -1).view(N, K // 128, 128).double()
    dense = ((q - w[2].double().view(N, -1, 1)) * w[1].double().view(N, -1, 1)).view(N, K)  # not rounded to bf16
    return w, dense


def _x(M, K):
    return torch.randn(M, K, device="cuda", generator=torch.Generator(device="cuda").manual_seed(M * K)).to(torch.bfloat16)


@pytest.mark.parametrize("N,K", [(16, 128), (48, 512), (528, 1664), (4112, 3968), (2048, 4608), (1040, 5504), (336, 11008), (4128, 8320),
                                 (8192, 2176), (8192, 512), (8224, 2688)])
def test_forward(hip_lib, N, K):
    from latentq_llm_amd import ops
    w, dense = _mat(N, K, N + K)
    for M in (1, 3, 4, 5, 8, 9, 12, 13, 16):
        x = _x(M, K)
        want = x.double() @ dense.t()
        y = ops.a16w4_forward(x, *w, (N, K))
        assert ((y.double() - want).norm() / want.norm()).item() < TOL, M
        assert torch.equal(ops.a16w4_forward(x, *w, (N, K)), y), M


@pytest.mark.parametrize("N,K", [(16, 128), (2048, 640), (4096, 2176), (4112, 1664), (8192, 2560), (6144, 4736), (8208, 1152), (9088, 3328),
                                 (11008, 4224)])
def test_gate_up(hip_lib, N, K):
    from latentq_llm_amd import ops
    (g, dg), (u, du) = _mat(N, K, 1), _mat(N, K, 2)
    for M in (1, 4, 6, 8, 11, 12, 16):
        x = _x(M, K)
        a = x.double() @ dg.t()
        want = torch.nn.functional.silu(a) * (x.double() @ du.t())
        h = ops.a16w4_gate_up_silu(x, g, u, (N, K))
        assert ((h.double() - want).norm() / want.norm()).item() < TOL, M
        assert torch.equal(ops.a16w4_gate_up_silu(x, g, u, (N, K)), h), M
