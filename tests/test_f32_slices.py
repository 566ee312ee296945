"""The slices of a row-major product's inner dimension do not depend on how a step's token count is rounded (host code: no GPU)."""
import pytest

from alice_llm_amd.engine.step import PROMPT_GRAPH_ROUND, PROMPT_GRAPH_TOKENS, _bucket
from alice_llm_amd.hip import ops


@pytest.mark.parametrize("N,K", [(2304, 2048), (2304, 9216), (2048, 2048), (4096, 2304), (512, 5000), (64, 9216), (2304, 513)])
def test_rounded_token_counts_have_the_slices_of_the_exact_ones(N, K):
    hint = lambda M: ops.linear_split_hint(M, N, K, ops.LAYOUT_ROW)       # noqa: E731
    for M in range(2, 700):
        assert hint(M) == hint(_bucket(M)), M
        if M <= PROMPT_GRAPH_TOKENS:
            assert hint(M) == hint(-(-M // PROMPT_GRAPH_ROUND) * PROMPT_GRAPH_ROUND), M
