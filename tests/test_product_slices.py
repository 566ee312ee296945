"""The slices of a fragment-layout product's inner dimension, and which kernel takes them (host code: no GPU)."""
import pytest
import torch

from alice_llm_amd.hip import ops
from alice_llm_amd.parts.base import FragmentActs

SIZES = [(12576, 4096), (12224, 4096), (2304, 2304), (2304, 9216), (3584, 14336), (2304, 2048), (2048, 8192), (2560, 1024), (3584, 4096), (4608, 36864)]


@pytest.mark.parametrize("N,K", SIZES)
def test_activations_that_stand_for_rows_have_the_slices_of_rows(N, K):
    w, differ = torch.empty(16, dtype=torch.bfloat16), 0
    for M in list(range(1, 130)) + list(range(433, 8200, 61)):
        row = ops.linear_split_hint(M, N, K, ops.LAYOUT_FRAG16, torch.empty(1, K, dtype=torch.bfloat16), w)
        flat = torch.empty(16, dtype=torch.bfloat16)
        if ops.linear_one_order(M, K):
            assert ops.linear_split_hint(M, N, K, ops.LAYOUT_FRAG16, FragmentActs(flat, M, K, as_rows=True), w) == row, M
        differ += ops.linear_split_hint(M, N, K, ops.LAYOUT_FRAG16, FragmentActs(flat, M, K), w) != row
    assert differ or (N, K) in [(2560, 1024)]           # (of so few inner elements neither order wants slices at many tokens)


@pytest.mark.parametrize("N,K", SIZES)
def test_a_product_takes_the_kernel_that_its_slices_were_proposed_for(N, K):
    for M in list(range(384, 1300, 16)) + list(range(433, 8200, 61)):
        split = ops.linear_split_hint(M, N, K, ops.LAYOUT_FRAG16)
        assert ops.linear_large_tile(M, N, K, split_k=split) == ops.linear_large_tile(M, N, K, split_k=0), (M, split)
