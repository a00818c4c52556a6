"""The forward of 17 to 64 tokens in one launch: rows on either side of every line between its forms (the waves of a workgroup and the
groups each has room for), of fewer groups than waves and of uneven numbers for them, and the sizes beside those of more than half of the
units' columns: fewer columns, and two rounds of them. Against the weights as they are in float64, with zeros that are no integers, too."""
import pytest
import torch

from tests.util import make_w4, randn_bf16, rel_l2

pytestmark = pytest.mark.gpu

SIZES = ([(M, 2064, 128 * G) for M in (17, 32) for G in (1, 7, 9, 32, 33, 63)] + [(M, 4080, 128 * G) for M in (18, 31) for G in (64, 65, 81, 90)]
         + [(M, 2064, 128 * G) for M in (33, 48) for G in (1, 31, 32, 33, 47, 63)] + [(M, 2064, 128 * G) for M in (49, 64) for G in (1, 34, 35, 36, 63)]
         + [(17, 1920, 2560), (32, 1024, 7936), (33, 1408, 1536), (45, 384, 5632), (48, 1920, 7936), (64, 2048, 1024), (40, 1152, 6784)]
         + [(17, 16, 128), (32, 2048, 2048), (31, 528, 11520), (48, 1040, 1152), (33, 144, 9216), (45, 2048, 5504), (48, 4096, 8192), (64, 16, 7168), (50, 2048, 5504), (49, 272, 128)]
         + [(17, 4112, 128), (25, 8192, 2048), (32, 5504, 2944)])


@pytest.mark.parametrize("M,N,K", SIZES)
def test_forward(hip_lib, M, N, K):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K)) == ("few_x16", 1, 0)
    codes, p, s, z = make_w4(N, K, M + N + K)
    z[::3] += 0.375
    w = ((codes.cuda().double().view(N, -1, 128) - z.cuda().double().view(N, -1, 1)) * s.cuda().double().view(N, -1, 1)).view(N, K)
    x, b = randn_bf16((M, K), M).cuda(), randn_bf16((N,), 1).cuda()
    want = x.double() @ w.t()
    dev = (p.cuda(), s.cuda(), z.cuda())
    # a result's own rounding to bf16 is 1.64e-3 to 1.67e-3 of the norm (2^-8 / sqrt(3) over the root mean square in a binade)
    assert rel_l2(ops.a16w4_forward(x, *dev, (N, K)), want) < 1.8e-3
    assert rel_l2(ops.a16w4_forward(x, *dev, (N, K), b), want + b.double()) < 1.8e-3


@pytest.mark.parametrize("M,N,K,kernel", [(33, 2048, 1024, "few_x16"), (33, 2048, 896, "few_x16"), (33, 2048, 2048, "few_x16"), (33, 2048, 2176, "few_x16"), (33, 1920, 4224, "few_x16"), (17, 2048, 2048, "few_x16"), (17, 2048, 2304, "few_x16"),
                                          (64, 1024, 6912, "few_x16"), (64, 1024, 7168, "few_x16"), (64, 1024, 7296, "staged_128x128"), (48, 1024, 7936, "few_x16"),
                                          (33, 16, 9216, "few_x16"), (48, 2048, 9344, "staged_128x128"), (17, 2048, 11520, "few_x16"), (17, 2048, 11648, "staged_128x128"),
                                          (48, 4096, 8192, "few_x16"), (48, 4080, 8192, "staged_128x128"), (49, 4096, 8192, "staged_128x128"),
                                          (32, 8192, 2048, "few_x16"), (32, 8208, 1024, "gemv_chunks"), (33, 4112, 1024, "staged_128x128"),
                                          (32, 4080, 11520, "few_x16"), (32, 4080, 11648, "staged_128x128"), (33, 4080, 8192, "staged_128x128")])
def test_lines_between_the_kernels(hip_lib, M, N, K, kernel):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, (N, K), compute_units=256)[0] == kernel
