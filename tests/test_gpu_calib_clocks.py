"""lq_calib_gemm_clocks: every kernel that it can run records four counters per workgroup, and nothing behind them."""
import ctypes

import pytest
import torch

from tests.util import make_w4, randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("backward,M,N,K,kernel", [(0, 64, 4096, 1024, "few_x16"), (0, 17, 4096, 4096, "few_x16"), (0, 45, 3088, 640, "few_x16"),
                                                   (0, 33, 11008, 384, "staged_128x128"), (0, 100, 1040, 896, "staged_128x128"),
                                                   (0, 256, 11008, 1024, "direct_128x128"), (0, 4224, 4096, 384, "staged_256x128"),
                                                   (1, 300, 1024, 2048, "staged_128x128")])
def test_every_workgroup_records(hip_lib, backward, M, N, K, kernel):
    from latentq_llm_amd import _C, ops
    assert ops.a16w4_plan(M, (N, K), backward=bool(backward), workspace_bytes=0)[0] == kernel
    _, p, s, z = (t.cuda() for t in make_w4(N, K, 1))
    a = randn_bf16((M, N if backward else K), 2).cuda()
    out = torch.empty((M, K if backward else N), dtype=torch.bfloat16, device="cuda")
    clocks = torch.full((1 << 16,), -1, dtype=torch.int64, device="cuda")
    count = ctypes.c_int64()
    _C.call("lq_calib_gemm_clocks", backward, a.data_ptr(), p.data_ptr(), s.data_ptr(), z.data_ptr(), out.data_ptr(), M, N, K, 128,
            clocks.data_ptr(), clocks.numel(), ctypes.addressof(count), torch.cuda.current_stream().cuda_stream)
    c = clocks.cpu()
    assert count.value > 0 and bool((c[4 * count.value:] == -1).all())
    t0, t1, r0, r1 = c[: 4 * count.value].view(-1, 4).unbind(1)
    assert bool((t0 > 0).all() and (t1 > t0).all() and (r0 > 0).all() and (r1 >= r0).all())
    want = ops.a16w4_dx(a, p, s, z, (N, K)) if backward else ops.a16w4_forward(a, p, s, z, (N, K))
    assert (out.float() - want.float()).norm() < 1e-2 * want.float().norm()
