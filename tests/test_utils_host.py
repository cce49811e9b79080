"""The FP8 cast helpers on host tensors: evaluated with torch alone, without the native libraries."""

import numpy as np
import pytest
import torch

from deepep_amd import _lib, utils
from oracle import quant as oquant


@pytest.fixture
def no_native(monkeypatch):
    def refuse():
        raise ImportError("not built")

    monkeypatch.setattr(_lib, "host", refuse)
    monkeypatch.setattr(_lib, "load", refuse)


@pytest.mark.parametrize("tokens,hidden", [(1, 128), (5, 384), (3, 200), (2, 7)])
def test_cast_back_of_host_tensors_needs_no_library(no_native, tokens, hidden):
    blocks = -(-hidden // 128)
    gen = torch.Generator().manual_seed(hidden)
    padded = torch.randn(tokens, blocks * 128, generator=gen).bfloat16()
    codes, scales = oquant.cast_to_fp8_torch(padded)
    want = oquant.cast_back(codes.view(torch.uint8).numpy(), scales.numpy())
    got = utils.per_token_cast_back(codes[:, :hidden].contiguous(), scales)
    assert got.dtype == torch.bfloat16
    np.testing.assert_array_equal(got.view(torch.int16).numpy().view(np.uint16), want[:, :hidden])


def test_cast_back_of_empty_host_tensors(no_native):
    empty = torch.empty((0, 256), dtype=torch.float8_e4m3fn)
    assert utils.per_token_cast_back(empty, torch.empty((0, 2))).shape == (0, 256)


def test_quantiser_names_what_is_wrong_with_a_host_tensor():
    with pytest.raises(AssertionError, match="2D"):
        utils.per_token_cast_to_fp8(torch.zeros(128, dtype=torch.bfloat16))
    with pytest.raises(ValueError):
        utils.per_token_cast_to_fp8(torch.zeros(2, 128, dtype=torch.bfloat16))
