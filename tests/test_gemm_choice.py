"""Which grouped GEMM kernel a forward takes (host arithmetic, no GPU needed): what the cost model picks for the sizes that its
rules were measured at, so that a change of its constants that moves one of them is seen."""

import pytest

from deepep_amd import ops

FEW, FEW_ONE_WAVE = (32, 4), (32, 1)


@pytest.mark.parametrize("sizes,first,second", [
    # tokens, hidden, intermediate, top-k, experts, local experts, shared experts
    ((512, 7168, 2048, 8, 256, 32, 0), FEW, FEW),                # decode: 16 rows for each of 32 experts
    ((16384, 7168, 2048, 8, 384, 6, 0), (192, 4), (128, 4)),     # one EP64 rank's share: 340 rows for each of 6
    ((777, 2880, 1408, 4, 32, 32, 1), (128, 4), (128, 4)),       # 97 rows for each of 32, and a shared one
    ((8192, 7168, 2048, 8, 32, 32, 0), (192, 4), (192, 4)),      # 2048 rows for each of 32
    ((24, 7168, 2048, 2, 2, 2, 0), FEW_ONE_WAVE, FEW_ONE_WAVE),  # two experts, 24 rows each: one-wave workgroups
    ((24, 1024, 512, 16, 16, 16, 0), FEW_ONE_WAVE, FEW_ONE_WAVE),
])
def test_kernels_of_known_sizes(sizes, first, second):
    assert ops.megamoe_gemm_choice(*sizes) == (first, second)


@pytest.mark.parametrize("sizes,first,second", [
    ((512, 7168, 2048, 8, 256, 32, 0), "few_rows", "few_rows"),
    ((16384, 7168, 2048, 8, 384, 6, 0), "column_waves", "paired"),
    ((777, 2880, 1408, 4, 32, 32, 1), "paired", "paired"),
    ((8192, 7168, 2048, 8, 32, 32, 0), "column_waves", "column_waves"),
    ((24, 7168, 2048, 2, 2, 2, 0), "one_wave", "one_wave"),
    ((24, 1024, 512, 16, 16, 16, 0), "one_wave", "few_rows"),    # k = 512 is short for the one without LDS
    ((5000, 7168, 2048, 1, 55, 55, 0), "paired_streamed", "paired_streamed"),  # 91 rows for each of 55, 850 and 425 MB of weights
    ((5000, 7168, 2048, 1, 16, 16, 0), "paired", "paired"),
    ((4096, 1280, 1280, 2, 4, 4, 0), "paired", "two_by_two"),
])
def test_kernels_by_name(sizes, first, second):
    assert ops.megamoe_gemm_kernels(*sizes) == (first, second)


@pytest.mark.parametrize("choice", [ops.megamoe_gemm_choice, ops.megamoe_gemm_kernels])
def test_choice_refuses_bad_sizes(choice):
    for bad in ((0, 1024, 512, 2, 8, 8), (8, 1024, 512, 2, 4, 8), (8, 1024, 512, 0, 8, 8), (8, 1024, 512, 2, 8, 8, -1)):
        with pytest.raises(ValueError, match="bad sizes"):
            choice(*bad)
