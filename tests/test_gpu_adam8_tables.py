"""The optimizer step of blocks of 2048 on few blocks, which compute what a stored moment contributes for each element, and on
many, which look it up by its code: tensors of more than two blocks to a compute unit against their parts of fewer, on either
side of the line, every mode, bit for bit. (The small form is compared with the tensor chain elsewhere.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu
K = 2048


@pytest.mark.parametrize("mode", ["direction", "param", "ratio", "sr", "w4", "w8"])
def test_many_blocks_equal_few(hip_lib, mode):
    from latentq_llm_amd import ops
    from latentq_llm_amd.quant import three_fold_curve_4bit
    from tests.util import make_w4
    curves = []
    for mu in (0, 1):
        p1, y1, p2, y2 = three_fold_curve_4bit(mu)
        curves.append((p1, y1, p2 - p1, y2, 8 - p2))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rows = [0, 2 * cus, 2 * cus + 1, 3 * cus + 3]  # the largest without tables, a block alone, the rest
    N = rows[-1]
    gen = torch.Generator().manual_seed(1)
    rand = lambda lo, hi: lo * (hi / lo) ** torch.rand(N, 1, generator=gen)
    state = {"s1": torch.randint(0, 256, (N, K), generator=gen).byte(), "s2": torch.randint(0, 256, (N, K), generator=gen).byte(),
             "q1": rand(1e-7, 1e-4), "q2": rand(1e-9, 1e-5)}
    state["m1"], state["m2"] = state["q1"] * 128, state["q2"] * 255  # second moments down to nothing
    grad = torch.randn(N, K, generator=gen).mul(1e-3).to(torch.bfloat16)
    grad[::7, ::5] = 0
    _, codes, scales, zeros = make_w4(N, K, 2)
    extra = {"codes": codes.view(N, K // 2), "scales": scales.view(N, -1), "zeros": zeros.view(N, -1),
             "codes8": torch.randint(-127, 128, (N, K), generator=gen).to(torch.int8), "qs": rand(1e-4, 1e-3).to(torch.bfloat16),
             "res": torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), generator=gen).to(torch.int32),
             "out": torch.randn(N, K, generator=gen).to(torch.bfloat16)}
    make = lambda a, b: {k: v[a:b].clone().cuda() for k, v in {**state, **extra, "grad": grad}.items()}

    def step(t, first):
        moments = (t["s1"], t["s2"], t["q1"], t["m1"], t["q2"], t["m2"], 0.9, 0.95, 1e-8)
        n = len(t["s1"])
        if mode in ("direction", "param"):
            ops.adam8_update(t["grad"], *moments, 1e-3, **{mode: t["out"]})
        elif mode == "ratio":
            t["out"] = ops.adam8_ratio(t["grad"], *moments)
        elif mode == "sr":
            t["codes"] = ops.adam8_update(t["grad"], *moments, 1e-3, requant=(t["codes"].view(-1), t["scales"].view(-1, 1), t["zeros"].view(-1, 1), (n, K),
                                                                              11, 7 + first * K // 8)).view(n, -1)
        elif mode == "w4":
            ops.adam8_latent_w4_step(t["grad"], t["codes"].view(-1), t["res"].view(-1), t["scales"].view(-1, 1), t["zeros"].view(-1, 1), (n, K),
                                     *moments[:6], *curves, *moments[6:], 1e-3)
        else:
            ops.adam8_latent_w8_step(t["grad"], t["codes8"], t["res"].view(-1), t["qs"], *moments[:6], *curves, *moments[6:], 1e-3)
        return t

    parts = [step(make(a, b), a) for a, b in zip(rows, rows[1:])]
    for end in (N, rows[2]):
        for k, v in step(make(0, end), 0).items():
            want = torch.cat([p[k].reshape(p["s1"].shape[0], -1) for p in parts])[:end]
            assert torch.equal(v.reshape(end, -1).view(torch.uint8), want.view(torch.uint8)), (end, k)
