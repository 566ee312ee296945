"""The slices of a row-major product's inner dimension do not depend on how a step's token count is rounded (host code: no GPU)."""
import pytest
import torch

from alice_llm_amd.engine.step import PROMPT_GRAPH_ROUND, PROMPT_GRAPH_TOKENS, _bucket
from alice_llm_amd.hip import ops
from alice_llm_amd.parts.base import Precision
from alice_llm_amd.parts.linear import Linear


@pytest.mark.parametrize("N,K", [(2304, 2048), (2304, 9216), (2048, 2048), (4096, 2304), (512, 5000), (64, 9216), (2304, 513)])
def test_rounded_token_counts_have_the_slices_of_the_exact_ones(N, K):
    hint = lambda M: ops.linear_split_hint(M, N, K, ops.LAYOUT_ROW)       # noqa: E731
    for M in range(2, 700):
        assert hint(M) == hint(_bucket(M)), M
        if M <= PROMPT_GRAPH_TOKENS:
            assert hint(M) == hint(-(-M // PROMPT_GRAPH_ROUND) * PROMPT_GRAPH_ROUND), M


# beyond 128 tokens the slices of the 32-bit instruction's own plan where it takes any (the thirds' number is another and measures slower)
@pytest.mark.parametrize("M,N,K,slices", [(500, 2304, 9216, 4), (256, 4608, 4096, 4), (1024, 3584, 4096, 2), (384, 2304, 9216, 7), (17, 3584, 4096, 8),
                                          (128, 4096, 2304, 4), (256, 4096, 2304, 4)])
@pytest.mark.parametrize("precision,x_dtype,w_dtype", [("float32", torch.float32, torch.bfloat16), ("bfloat16", torch.bfloat16, torch.float32)])
def test_slices_of_products_with_a_bfloat16_operand(monkeypatch, M, N, K, slices, precision, x_dtype, w_dtype):
    """A bfloat16 checkpoint on the 32-bit path, and 32-bit weights kept as stored on the bfloat16 path."""
    asked = []
    monkeypatch.setattr(ops, "linear", lambda *a, split_k, **k: asked.append(split_k))
    part = Linear(K, N, Precision.of(precision, keep_stored=True))
    part.load(torch.empty(N, K, dtype=w_dtype))
    part(torch.empty(M, K, dtype=x_dtype), torch.float32, allow_partials=True)
    assert part.layout == ops.LAYOUT_ROW and asked == [slices]


def test_slices_of_32_bit_operands_that_are_not_aligned(monkeypatch):
    """Rows that are no multiple of 16 bytes, and rows that do not start at one, stay with the 32-bit instruction and its slices."""
    asked = []
    monkeypatch.setattr(ops, "linear", lambda *a, split_k, **k: asked.append(split_k))
    M, N, K = 256, 4096, 2304
    for at, columns in ((0, K), (1, K), (0, K + 1)):
        part = Linear(columns, N, Precision.of("float32"))
        part.load(torch.empty(N, columns))
        part(torch.empty(M * columns + 1)[at:at + M * columns].view(M, columns), torch.float32, allow_partials=True)
    assert asked == [4, 1, 1]
