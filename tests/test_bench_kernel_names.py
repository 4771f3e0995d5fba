"""The kernel that the benchmark's records name is the one that the library's
automatic choice takes (make_logistic in csrc/logistic.hip)."""
import pytest

import bench


@pytest.mark.parametrize("x_dtype, N, D, C, name", [
    ("fp8", 2_000_000, 256, 64, "logit_split_kernel<256, fp8>"),
    ("fp8", 65_536, 33, 17, "logit_split_kernel<64, fp8>"),
    ("fp8", 65_536, 33, 16, "logit_partial_f32<XFP8>"),
    ("fp8", 65_535, 33, 1024, "logit_partial_f32<XFP8>"),
    ("fp8", 100_000, 257, 1024, "logit_partial_f32<XFP8>"),
    ("fp32", 1000, 26, 4, "persistent_head_kernel<LogisticChainModel<32>>"),
    ("fp32", 3999, 200, 4, "logit_partial_f32 (VALU tile)"),
    ("fp32", 15_999, 70, 9, "logit_partial_f32 (VALU tile)"),
    ("fp32", 1_000_000, 16, 17, "logit_partial_f32 (VALU tile)"),
    ("fp32", 581_012, 55, 1, "logit_rows_kernel<1, 1>"),
    ("fp32", 1_000_000, 256, 31, "logit_rows_kernel<4, 4>"),
    ("fp32", 1_000_000, 130, 8, "logit_rows_kernel<3, 2>"),
    ("fp32", 1_000_000, 257, 31, "logit_partial_f32 (VALU tile)"),
    ("fp32", 1_000_000, 257, 40, "logit_partial_f32 (VALU tile)"),
    ("fp32", 581_012, 55, 32, "logit_partial_f32 or logit_split_kernel<64, fp32>"),
    ("fp32", 581_012, 55, 129, "logit_split_kernel<64, fp32>"),
    ("bf16", 2_000_000, 256, 1024, "logit_bf16_pipe<256, true>"),
])
def test_names_follow_the_automatic_choice(x_dtype, N, D, C, name):
    assert bench.model_kernel_name(x_dtype, N, D, C, single=True).startswith(name)
