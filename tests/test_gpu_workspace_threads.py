"""Scratch buffers of host threads that share a stream: each thread has its own, and their number stays bounded."""
import threading

import pytest
import torch

from tests.util import make_w4, randn_bf16

pytestmark = pytest.mark.gpu


def test_threads_on_one_stream(hip_lib):
    from latentq_llm_amd import ops
    x = randn_bf16((45, 4096), 1).cuda()
    mine = ops._workspace(x, 45, 4096)[0]
    assert ops._workspace(x, 45, 4096)[0] is mine
    other, errors = [], []
    both = threading.Barrier(2, timeout=60)  # a thread that ended may leave its number, and the buffer with it, to the next
    mats = [tuple(t.cuda() for t in make_w4(2048, 4096, seed)[1:]) for seed in (2, 3)]
    want = [(ops.a16w4_forward(x, *m, (2048, 4096)), ops.a16w4_gate_up_silu(x, m, mats[0], (2048, 4096))) for m in mats]

    def work(i):
        try:
            other.append(ops._workspace(x, 45, 4096)[0])
            both.wait()
            for _ in range(50):
                y, h = ops.a16w4_forward(x, *mats[i], (2048, 4096)), ops.a16w4_gate_up_silu(x, mats[i], mats[0], (2048, 4096))
                assert torch.equal(y, want[i][0]) and torch.equal(h, want[i][1])
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert len({b.data_ptr() for b in other + [mine]}) == 3
    for _ in range(2 * ops.WORKSPACE_MAX_STREAMS):
        t = threading.Thread(target=ops._workspace, args=(x, 45, 4096))
        t.start()
        t.join()
    assert len([k for k in ops._WORKSPACE if k[0] == torch.cuda.current_device()]) <= ops.WORKSPACE_MAX_STREAMS
