"""When the keys of a prompt's longest tiles are cut, and that a step works it out once (host code: no GPU)."""
from types import SimpleNamespace

import pytest
import torch

from alice_llm_amd.engine.step import StepContext
from alice_llm_amd.hip import ops


# several sequences (the rule knows the longest alone) and windows must promise more: measured uncut and cut 107 and 113 us, 50.7 and 53.1,
# 97.7 and 101, 162.5 and 167.9, 162.8 and 167.1; the last three 57.8 and 46, 66.7 and 48, 34.5 and 34
@pytest.mark.parametrize("n,new,context,heads,window,cuts", [
    (2, 2000, 2500, (8, 4), None, False), (2, 1500, 1500, (8, 8), 1024, False), (2, 2000, 2500, (8, 8), None, False),
    (1, 5000, 5000, (8, 1), 4096, False), (1, 5000, 5000, (8, 2), 4096, False),
    (1, 2048, 2048, (8, 4), None, True), (2, 1500, 1500, (8, 4), None, True)])
def test_what_loses_is_not_cut(n, new, context, heads, window, cuts):
    assert (ops.prefill_cut(n, new, context, *heads, 256, window) > 1) == cuts


def context(**sizes):
    places = {name: {} for name in StepContext.__dataclass_fields__ if name in ("cuts", "arrivals")}
    assert set(places) == {"cuts", "arrivals"}
    return SimpleNamespace(**sizes, **places)


def test_a_step_works_it_out_once_and_keeps_counts_of_their_own_for_each_stream(monkeypatch):
    asked, stream = [], [11]
    rule = ops.prefill_cut
    monkeypatch.setattr(ops, "prefill_cut", lambda *sizes: asked.append(sizes) or rule(*sizes))
    monkeypatch.setattr(ops, "_stream", lambda: stream[0])
    ctx, heads = context(n_seqs=1, max_new=2048, max_context=2048), (8, 4, 256)
    cut, whole = ops._cut_of(ctx, *heads, None, "cpu")
    assert cut > 1 and whole.numel() == ops.prefill_counts(1, 2048, 2048, *heads, None, cut) and not whole.any()
    for _ in range(3):
        again = ops._cut_of(ctx, *heads, None, "cpu")
        assert again[0] == cut and again[1] is whole and len(asked) == 1
    # a layer whose window asks for more counts, and then the first again
    cut_w, grown = ops._cut_of(ctx, *heads, 1900, "cpu")
    assert cut_w > 1 and grown.numel() > whole.numel() and not grown.any()
    assert ops._cut_of(ctx, *heads, None, "cpu")[1] is grown and len(asked) == 2
    assert ops._cut_of(ctx, *heads, 1024, "cpu") == (1, None)
    stream[0] = 12
    assert ops._cut_of(ctx, *heads, None, "cpu")[1] is not grown
    bare = SimpleNamespace(n_seqs=1, max_new=2048, max_context=2048)     # a context of somebody else's
    assert ops._cut_of(bare, *heads, None, "cpu")[0] == cut and not hasattr(bare, "arrivals")
