"""The kernels and tiles that products take, at sizes where a choice by the step times alone, or by one set of constants for two kernels,
or a line drawn from too few sizes, took one that is 2 % slower and more. Host arithmetic for 256 compute units, no launch."""
import pytest


# (store, add or int8), tokens, [N, K]; us on 128 x 128 / 192 x 256 / 256 x 256
@pytest.mark.parametrize("form,M,shape,tile", [
    ("store", 13, (4096, 4096), (256, 256, 8)),     # 11.9 / 13.9 / 10.9
    ("store", 20, (6400, 2304), (256, 256, 8)),     # 11.1 / 13.7 / 10.3
    ("store", 2956, (11008, 3584), (256, 256, 4)),  # 229 / 231 / 213
    ("store", 256, (8576, 2304), (192, 256, 8)),    # 24.3 / 20.4 / 22.8
    ("add", 3316, (3584, 11008), (256, 256, 4)),    # 262 / 266 / 242
    ("int8", 64, (3584, 8832), (256, 256, 8)),      # 41.5 / 44.3 / 39.1
    ("int8", 25, (5888, 2816), (256, 256, 8)),      # 22.8 / 31.0 / 21.7
])
def test_weight_gradient(hip_lib, form, M, shape, tile):
    from latentq_llm_amd import ops
    assert ops.weight_grad_plan(form, M, shape, 256) == tile


# two products into one input gradient are planned as one of twice the rows of W; us on 128 / 192 / 256 rows
@pytest.mark.parametrize("M,shape,kernel,cut", [
    (256, (10752, 4096), "staged_256x128", True),   # int8 39.6 / 44.7 / 36.0
    (640, (22016, 3072), "staged_256x128", True),   # pair 123 / 128 / 112
    (832, (17408, 2304), "staged_256x128", True),   # pair 99.3 / 100 / 90.9
    (601, (8064, 2304), "staged_256x128", True),    # 42.6 / 40.4 / 39.6
    (3461, (4096, 1024), "staged_128x128", False),  # int8 37.6 / 43.0 / 50.5 whole, 41.0 in slices of 256 rows
    (1664, (4352, 2048), "staged_128x128", False),  # 39.3 / 45.6 / 51.7 whole, 42.0 in slices of 256 rows
])
def test_input_gradient(hip_lib, M, shape, kernel, cut):
    from latentq_llm_amd import ops
    got, slices, _ = ops.a16w4_plan(M, shape, backward=True, compute_units=256)
    assert (got, slices > 1) == (kernel, cut)


# with the SiLU backward behind it; us on 128 / 192 / 256 rows
@pytest.mark.parametrize("M,shape", [(3462, (3840, 7936)),   # 266 / 265 / 255
                                     (1728, (4096, 11008)),  # 195 / 203 / 187
                                     (2432, (3840, 11008))])  # 253 / 257 / 245
def test_input_gradient_with_silu(hip_lib, M, shape):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, shape, silu=True, compute_units=256) == ("staged_256x128", 1, 0)


# gate / up of 49 to 64 tokens; us in slices of K / in one launch
@pytest.mark.parametrize("M,shape", [(54, (3584, 6144)),   # 17.2 / 18.8
                                     (62, (2336, 5888)),   # 17.3 / 18.0
                                     (50, (4096, 5888))])  # 17.2 / 18.9
def test_gate_up_on_a_long_k(hip_lib, M, shape):
    from latentq_llm_amd import ops
    kernel, _, slices = ops.a16w4_gate_up_plan(M, shape, compute_units=256)
    assert kernel == "staged_128x128" and slices > 1
    assert ops.a16w4_gate_up_plan(M, shape, workspace_bytes=0, compute_units=256)[0] == "few_x16"  # K cannot be cut


# forward of 17 to 128 tokens, most on half of the units' columns and fewer; us otherwise / in one launch (36 tokens in the place of 33 and so on)
@pytest.mark.parametrize("M,shape", [(45, (2048, 4096)),   # 10.6 / 6.9
                                     (33, (2048, 2304)),   # 9.3 / 5.0
                                     (64, (2048, 7040)),   # 13.5 / 12.0
                                     (24, (2048, 2048)),   # 6.8 / 4.4
                                     (17, (1024, 1024)),   # 6.1 / 3.4
                                     (45, (4096, 8192)),   # 15.6 / 13.3
                                     (80, (1536, 1920)),   # 8.8 / 6.5
                                     (100, (1040, 1664))])  # 8.6 / 7.8
def test_forward_of_few_columns(hip_lib, M, shape):
    from latentq_llm_amd import ops
    assert ops.a16w4_plan(M, shape, compute_units=256) == ("few_x16", 1, 0)


# gate / up of 17 to 64 tokens on 8 columns a unit and fewer
@pytest.mark.parametrize("M,shape", [(20, (2048, 1536)),   # 8.7 / 4.9
                                     (45, (1408, 4096))])  # 14.3 / 9.6
def test_gate_up_of_few_columns(hip_lib, M, shape):
    from latentq_llm_amd import ops
    assert ops.a16w4_gate_up_plan(M, shape, compute_units=256)[0] == "few_x16"


def test_weight_gradient_plan_refuses_what_the_product_does(hip_lib):
    from latentq_llm_amd import ops
    from latentq_llm_amd._C import LatentQError
    for form, shape, text in (("store", (100, 128), "multiple of 8"), ("int8", (128, 136), "K=136 of 16"), ("add", (0, 128), "positive")):
        with pytest.raises(LatentQError, match=text):
            ops.weight_grad_plan(form, 64, shape, 256)
