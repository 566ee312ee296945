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


# sums without an epilogue: below 448 tokens no tile of 256 tokens; a round of blocks that loses to the tiled kernel on weights that no cache
# holds; sizes that gain by a tenth and more (the 2B, 9B and 27B widths)
@pytest.mark.parametrize("M,N,K,takes", [(447, 4608, 36864, False), (450, 4608, 36864, True), (1024, 2304, 2048, False), (505, 3584, 4096, False),
                                         (768, 2048, 8192, False), (1536, 4608, 4096, False), (2048, 2304, 9216, True), (1024, 3584, 14336, True),
                                         (4096, 3584, 4096, True), (8192, 2304, 2048, True), (2048, 2304, 9216 + 32, False)])
def test_where_the_tiles_of_256_tokens_begin(M, N, K, takes):
    assert bool(ops.linear_large_tile(M, N, K, split_k=0)) == takes


@pytest.mark.parametrize("M,takes", [(447, False), (448, True), (2048, True)])
def test_gated_products_take_them_too(M, takes):
    for form in (0.0, ops.GATED_SILU):
        assert bool(ops.linear_large_tile(M, 9216, 2304, epilogue=ops.EPI_GEGLU, epi_param=form, dtype=torch.bfloat16)) == takes
    assert not ops.linear_large_tile(M, 9216, 2304, epilogue=ops.EPI_GEGLU, epi_param=7.0, dtype=torch.bfloat16)      # the limited form
    assert not ops.linear_large_tile(M, 9216, 2304, epilogue=ops.EPI_GEGLU)                                            # 32-bit output
