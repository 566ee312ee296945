"""Prompt attention with a tile's keys cut over several blocks: every head grouping, prefixes, windows, sinks, more parts than blocks of keys."""
import pytest
import torch

from alice_llm_amd.engine.step import StepContext
from alice_llm_amd.hip import ops
from test_gpu_kernels import DEV, acts_from_fragments, close, frag_case

pytestmark = pytest.mark.gpu


# heads a block: 2, 4, 1 and 2 (the last in three passes over a group of 6); one sequence, sequences of unlike lengths, tokens after a prefix
@pytest.mark.parametrize("nH,nKV", [(8, 4), (8, 2), (3, 3), (12, 2)])
@pytest.mark.parametrize("cap,window", [(None, None), (5.0, 50), (50.0, 300)])
@pytest.mark.parametrize("lens,new", [((300,), (300,)), ((150, 64, 33), (20, 3, 33)), ((700, 40), (333, 1))])
def test_cut_keys(nH, nKV, cap, window, lens, new):
    q, kp, vp, bt, cu, ctx, ref, scale = frag_case(nH, nKV, 256, lens, new, cap, window, seed=3)
    kw = dict(num_heads=nH, n_seqs=len(lens), max_new=max(new), max_context=max(lens), scale=scale, softcap=cap, window=window)
    sink = torch.linspace(-3, 4, nH, device=DEV)
    for s in (None, sink):
        whole = torch.full_like(q, float("nan"))
        ops.attention_prefill(q, kp, vp, whole, cu, ctx, bt, variant=ops.PREFILL_SHARED8, sink=s, **kw)
        for cut in (2, 3, 8):
            n = ops.prefill_counts(len(lens), max(new), max(lens), nH, nKV, 256, window, cut)
            arrivals = torch.zeros(n, dtype=torch.int32, device=DEV)
            outs = []
            for _ in range(3):                                # the counts are left as they were found, whoever comes last
                out = torch.full_like(q, float("nan"))
                ops.attention_prefill(q, kp, vp, out, cu, ctx, bt, cut=cut, arrivals=arrivals, sink=s, **kw)
                outs.append(out)
            assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]) and not arrivals.any()
            # a step of the result's rounding to bfloat16 (2^-7 of it), and weights that are rounded to bfloat16 for another
            # maximum: at most 2^-8 of each, of values up to 4.5
            close(out, whole.double(), 4.5 * 2 ** -8, 2 ** -7)
            if s is None:
                close(out, ref, 2e-2)
                assert (out.double().cpu() - ref).norm() <= 1.02 * (whole.double().cpu() - ref).norm()
            flat = torch.full(((-(-q.shape[0] // 16) * 16) * nH * 256,), float("nan"), dtype=torch.bfloat16, device=DEV)
            ops.attention_prefill(q, kp, vp, flat, cu, ctx, bt, cut=cut, arrivals=arrivals, sink=s, out_layout=ops.LAYOUT_FRAG16, **kw)
            assert torch.equal(acts_from_fragments(flat, q.shape[0], nH * 256), out.cpu())


def test_what_is_cut():
    """The rule's edges, and what is refused."""
    assert ops.prefill_cut(1, 2048, 2048, 8, 4, 256, None) > 1 and ops.prefill_cut(1, 640, 2640, 8, 4, 256, None) > 1
    assert ops.prefill_cut(1, 2048, 2048, 32, 16, 128, None) == 1         # heads of 128
    assert ops.prefill_cut(1, 256, 8192, 8, 4, 256, None) == 1            # may be captured
    assert ops.prefill_cut(16, 2048, 2048, 16, 8, 256, None) == 1         # blocks enough
    assert ops.prefill_cut(1, 2048, 100, 8, 4, 256, None) == 1 and ops.prefill_cut(0, 0, 0, 8, 4, 256, None) == 1
    q, kp, vp, bt, cu, ctx, ref, scale = frag_case(8, 4, 256, (300,), (300,), None, None, seed=3)
    kw = dict(num_heads=8, n_seqs=1, max_new=300, max_context=300, scale=scale, softcap=None, window=None, cut=2)
    n = ops.prefill_counts(1, 300, 300, 8, 4, 256, None, 2)
    with pytest.raises(ops.HipLibraryError):
        ops.attention_prefill(q, kp, vp, torch.empty_like(q), cu, ctx, bt, arrivals=torch.zeros(n - 1, dtype=torch.int32, device=DEV), **kw)
    with pytest.raises(ops.HipLibraryError):
        ops.attention_prefill(q, kp, vp, torch.empty_like(q), cu, ctx, bt, arrivals=torch.zeros(n, dtype=torch.int32, device=DEV),
                              variant=ops.PREFILL_SHARED8, **kw)


# a whole prompt, tokens after a prefix, and two sequences of unlike lengths; a window that asks for other counts than none does
@pytest.mark.parametrize("lens,new,windows", [((2048,), (2048,), (None, 1900)), ((2640,), (640,), (None,)), ((1500, 900), (1000, 450), (None, 800))])
def test_layers_of_a_step(lens, new, windows):
    """The path of a model's layers: the step picks the cut and keeps the counts, which a layer with more of them replaces."""
    nH, nKV, d = 8, 4, 256
    sizes = (len(lens), max(new), max(lens), nH, nKV, d)
    counts = {w: ops.prefill_counts(*sizes, w, ops.prefill_cut(*sizes, w)) for w in windows if ops.prefill_cut(*sizes, w) > 1}
    assert len(set(counts.values())) == len(windows)         # all are cut, with unlike numbers of counts
    none = torch.empty(0, dtype=torch.int32, device=DEV)
    ctx = None
    for w in sorted(counts, key=counts.get) * 2:             # the fewest first: the second layer's counts are new ones
        q, kp, vp, bt, cu, ctxl, ref, scale = frag_case(nH, nKV, d, lens, new, 50.0, w, seed=5, dense=True)
        if ctx is None:
            ctx = StepContext(tokens=none, positions=none, seq_of_token=none, slots=none, want_rows=None, cu_seqlens=cu, context_lens=ctxl,
                              n_tokens=sum(new), n_seqs=len(lens), is_decode=False, max_new=max(new), max_context=max(lens),
                              max_position=max(lens) - 1)
        whole, out = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
        ops.attention_prefill(q, kp, vp, whole, cu, ctxl, bt, variant=ops.PREFILL_SHARED8, num_heads=nH, n_seqs=len(lens), max_new=max(new),
                              max_context=max(lens), scale=scale, softcap=50.0, window=w)
        ops.attention(q, kp, vp, out, ctx, bt, num_heads=nH, scale=scale, softcap=50.0, window=w, full_precision=False, kv_layout=ops.KV_FRAGMENT)
        close(out, whole.double(), 4.5 * 2 ** -8, 2 ** -7)   # (the bound of the test above)
        close(out, ref, 2e-2)
        assert not torch.equal(out, whole)                   # it is the cut form that ran
        (kept,) = ctx.arrivals.values()
        assert kept.numel() >= counts[w] and not kept.any()
    assert kept.numel() == max(counts.values()) and len(ctx.cuts) == len(windows)
