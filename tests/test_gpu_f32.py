"""The kernels of the true 32-bit path against 64-bit references: products and attention on the 32-bit matrix instruction, at
the edges of their tiles, slices and splits."""
import math
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

from alice_llm_amd.hip import ops
from helpers import TINY, random_tokens
from plain import gemma2_plain as P
from test_gpu_kernels import DT, attention_case, close, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"


# ------------------------------------------------------------------ products
@pytest.mark.parametrize("M,N,K", [(1, 64, 9216), (4, 16400, 72), (9, 64, 32), (13, 46, 1032), (3, 70, 33), (8, 2304, 2305), (16, 40, 9220), (5, 24, 30), (16, 100, 2048), (17, 64, 40), (31, 33, 36), (33, 65, 68), (64, 128, 31), (129, 257, 96), (250, 2304, 2048), (500, 1000, 2308),
                                   (257, 4002, 100), (250, 8202, 36), (250, 24004, 36)])
@pytest.mark.parametrize("xdt,wdt", [("float32", "float32"), ("float32", "bfloat16"), ("bfloat16", "float32")])
def test_products_at_the_edges_of_tiles_and_slices(M, N, K, xdt, wdt):
    x, w = rnd(M, K, seed=M, dtype=DT[xdt]), rnd(N, K, seed=N, scale=0.1, dtype=DT[wdt])
    # K roundings of at most 2^-24 of a partial sum of size 0.1 sqrt(K) add up to 0.1 K 2^-24; eight times that over all elements
    ref, tol = x.double() @ w.double().T, 8 * 0.1 * K * 2 ** -24
    full = xdt == "float32"
    y = torch.empty(M, N, device=DEV)
    ops.linear(x, w, y, n_out=N, k_in=K, full_precision=full)
    close(y, ref, tol)
    for split in {2, 3, 8, ops.linear_split_hint(M, N, K, ops.LAYOUT_ROW)}:
        parts = torch.full((split, M, N), float("nan"), device=DEV) if split > 1 else torch.empty(M, N, device=DEV)
        ops.linear(x, w, parts, n_out=N, k_in=K, split_k=split, full_precision=full)
        close(parts.sum(0) if split > 1 else parts, ref, tol)
    if N % 2 == 0:
        out = torch.empty(M, N // 2, device=DEV)
        ops.linear(x, w, out, n_out=N // 2, k_in=K, epilogue=ops.EPI_GEGLU, full_precision=True)
        g, u = ref[:, :N // 2], ref[:, N // 2:]
        close(out, F.gelu(g, approximate="tanh") * u, 4 * tol, 1e-5)


@pytest.mark.parametrize("M", [1, 2, 16, 40])
@pytest.mark.parametrize("K", [64, 4, 31, 97, 4101])
def test_products_of_rows_that_are_not_aligned(M, K):
    big = rnd(M * K + 1, seed=3)
    for dt in (torch.float32, torch.bfloat16):
        x, w = big[1:].view(M, K), rnd(48 * K + 3, seed=4).to(dt)[3:].view(48, K)
        ref = x.double() @ w.double().T
        for split in (1, 2, 8):
            y = torch.empty(*((split,) if split > 1 else ()), M, 48, device=DEV)
            ops.linear(x, w, y, n_out=48, k_in=K, split_k=split, full_precision=True)
            close(y.sum(0) if split > 1 else y, ref, 8 * K * 2 ** -24)


@pytest.mark.parametrize("N,K", [(64, 4101), (2304, 2305), (48, 20), (16400, 37)])
def test_a_few_tokens_give_each_what_one_of_them_gives(N, K):
    """Rows of any length, up to 16 tokens: a token's sums are added in the same order however many there are."""
    x, w = rnd(16, K, seed=1), rnd(N, K, seed=2)
    outs = []
    for M in (2, 5, 16):
        outs.append(torch.empty(M, N, device=DEV))
        ops.linear(x[:M].contiguous(), w, outs[-1], n_out=N, k_in=K, full_precision=True)
    assert torch.equal(outs[0], outs[2][:2]) and torch.equal(outs[1], outs[2][:5])


def test_products_refuse_slices_with_an_epilogue_and_too_many():
    x, w = rnd(16, 64), rnd(64, 64)
    with pytest.raises(ops.HipLibraryError, match="partial sums"):
        ops.linear(x, w, torch.empty(2, 16, 64, device=DEV), n_out=64, k_in=64, epilogue=ops.EPI_SOFTCAP, epi_param=1.0, split_k=2, full_precision=True)
    with pytest.raises(ops.HipLibraryError, match="slices"):
        ops.linear(x, w, torch.empty(9, 16, 64, device=DEV), n_out=64, k_in=64, split_k=9, full_precision=True)


def test_sliced_products_add_in_one_order_in_captured_and_eager_steps():
    """A layer whose output and down projections go in slices (which the tiny shapes are too narrow for): prompts whose token
    count a captured step rounds up, and single tokens of 33 sequences, for which it takes 64 rows: the same bits."""
    import alice_llm_amd as alice
    raw = dict(TINY["tiny-a"][0], num_hidden_layers=1, hidden_size=2304, num_attention_heads=8, num_key_value_heads=4, head_dim=256,
               intermediate_size=1024, query_pre_attn_scalar=256)
    model = alice.Model.random(raw, seed=4, dtype="float32", fast=True)
    eager, graph = (model.engine(max_tokens=64 * 70, max_seqs=40, use_graphs=g) for g in (False, True))
    assert graph.capture_prompts
    assert ops.linear_split_hint(49, 2304, 2048, ops.LAYOUT_ROW) > 1
    for n in (49, 129, 200):
        for seed in range(3):                                            # seen, captured, replayed
            toks = random_tokens(256, n, seed)
            a, b = ([e.open(1), e] for e in (eager, graph))
            assert torch.equal(a[1].step(a[0], [toks], "last"), b[1].step(b[0], [toks], "last")), (n, seed)
            eager.close(a[0]), graph.close(b[0])
    slots = [e.open(33) for e in (eager, graph)]
    first = [random_tokens(256, 2, 100 + i) for i in range(33)]
    logits = [e.step(s, first, "last") for e, s in zip((eager, graph), slots)]
    for _ in range(3):
        ids = [[int(t)] for t in logits[0].argmax(dim=1)]
        logits = [e.step(s, ids, "last") for e, s in zip((eager, graph), slots)]
        assert torch.equal(*logits)


@pytest.mark.parametrize("family", ["novotar", "vazilorn"])
def test_sliced_products_through_the_residual_adds(family, monkeypatch):
    """Down projections in slices ahead of an add of several branches (from 256 rows on) and of one with a norm element by element:
    prompts and single tokens of a batch, against the plain model."""
    import helpers
    from test_gpu_novotar import assert_close
    from plain import novotar_plain, vazilorn_plain
    raw = {"novotar": helpers._nv_c, "vazilorn": helpers._vz_a}[family]()
    for layer in raw["layers"]:
        if layer["mlp"] is not None and layer["mlp"]["kind"] == "dense":
            layer["mlp"] = dict(layer["mlp"], ff=2048)
    cfg, t = {"novotar": helpers.novotar_tensors, "vazilorn": helpers.vazilorn_tensors}[family](raw, 5)
    plain = {"novotar": novotar_plain.PlainNovotar, "vazilorn": vazilorn_plain.PlainVazilorn}[family](raw, {k: v.double() for k, v in t.items()})
    model = helpers.model_from_tensors(cfg, {k: v.to(DEV) for k, v in t.items()}, "float32")
    added, old = set(), {}
    for name in ("add_branches", "add_dyntanh"):
        old[name] = getattr(ops, name)
    monkeypatch.setattr(ops, "add_branches", lambda x, many, *a, **k: (added.update(("many", b[0].shape[0]) for b in many if b[0].dim() == 3),
                                                                       old["add_branches"](x, many, *a, **k)))
    monkeypatch.setattr(ops, "add_dyntanh", lambda *a, **k: (added.add(("pointwise", k.get("n_partials", 1))), old["add_dyntanh"](*a, **k)))
    toks = [random_tokens(raw["vocab"], n, n) for n in (70, 300, 9)]
    refs = [plain.forward(x) for x in toks]
    eng = model.engine(max_tokens=64 * 16, max_seqs=3)
    for x, ref in zip(toks, refs):
        s = eng.open(1)
        assert_close(eng.step(s, [x], "all"), ref, "float32", len(x))
        eng.close(s)
    slots = eng.open(3)
    got = [eng.step(slots, [x[:-2] for x in toks], "last")] + [eng.step(slots, [[x[j]] for x in toks], "last") for j in (-2, -1)]
    for i, ref in enumerate(refs):
        assert_close(torch.stack([g[i] for g in got]), ref[-3:], "float32", i)
    kind = {"novotar": "many", "vazilorn": "pointwise"}[family]
    assert any(k == kind and n > 1 for k, n in added)


# ------------------------------------------------------------------ attention
def ctx_of(lens, new, pos, seq):
    cu = [0]
    for n in new:
        cu.append(cu[-1] + n)
    return SimpleNamespace(positions=pos, seq_of_token=seq, cu_seqlens=torch.tensor(cu, dtype=torch.int32, device=DEV), n_seqs=len(new),
                           is_decode=max(new) == 1, max_context=max(lens), max_position=max(lens) - 1, rounded_seqs=len(new),
                           rounded_context=max(lens))


@pytest.mark.parametrize("nH,nKV,d", [(4, 1, 64), (6, 2, 128), (8, 4, 256), (5, 5, 64), (16, 1, 128)])
@pytest.mark.parametrize("cap,window", [(None, None), (5.0, 50), (50.0, 7), (None, 16)])
def test_attention_prompts_pieces_and_single_tokens(nH, nKV, d, cap, window):
    for lens, new in (((5, 130, 66), (5, 130, 66)), ((200, 1, 77, 16), (1, 1, 1, 1)), ((150, 64, 33), (20, 3, 1))):
        q, kp, vp, bt, pos, seq, ref, scale = attention_case("float32", nH, nKV, d, lens, new, cap, window, seed=3)
        for splits in (None, 1, 2, 5):
            out = torch.full_like(q, float("nan"))
            ops.attention_f32(q, kp, vp, out, ctx_of(lens, new, pos, seq), bt, num_heads=nH, scale=scale, softcap=cap, window=window, splits=splits)
            close(out, ref, 1e-5)


def test_attention_keeps_values_that_are_no_numbers_to_the_queries_that_see_them():
    """The value at position 37 is infinite and the one at 70 not a number: rows before see neither, rows behind the window
    of 20 neither again, whatever tile of 16 keys or queries they share."""
    nH, nKV, d, L, window = 4, 2, 64, 96, 20
    q, kp, vp, bt, pos, seq, _, scale = attention_case("float32", nH, nKV, d, (L,), (L,), None, window, seed=8)
    for at, what in ((37, math.inf), (70, math.nan)):
        vp[int(bt[0, at // 64]), :, at % 64, 3] = what
    rows = lambda pool: torch.cat([pool[int(bt[0, i])] for i in range(2)], dim=1)[:, :L].transpose(0, 1).double().cpu()   # noqa: E731
    ref = P.attention_core(q.view(L, nH, d).double().cpu(), rows(kp), rows(vp), scale, None, window)
    for splits in (1, 2):
        out = torch.empty_like(q)
        ops.attention_f32(q, kp, vp, out, ctx_of((L,), (L,), pos, seq), bt, num_heads=nH, scale=scale, softcap=None, window=window, splits=splits)
        got = out.view(L, nH, d).double().cpu()
        fine = torch.isfinite(ref)
        assert not fine[37:57, :, 3].any() and fine[:37].all() and torch.equal(fine, torch.isfinite(got))
        assert (got - ref)[fine].abs().max() < 1e-5


@pytest.mark.parametrize("at", [0, 15, 16, 40, 64])
def test_attention_keeps_a_score_that_is_no_number(at):
    """A key that is not a number: every query that sees it gets none, also where it is the one key of its tile that the query sees;
    the queries before it and those behind the window see nothing of it.  As prompts, and the last positions as single tokens."""
    nH, nKV, d, L, window = 4, 2, 64, 80, 30
    q, kp, vp, bt, pos, seq, _, scale = attention_case("float32", nH, nKV, d, (L,), (L,), None, window, seed=8)
    kp[int(bt[0, at // 64]), :, at % 64, 5] = math.nan
    sees = torch.tensor([at <= i < at + window for i in range(L)])
    for splits in (1, 2, 3):
        out = torch.empty_like(q)
        ops.attention_f32(q, kp, vp, out, ctx_of((L,), (L,), pos, seq), bt, num_heads=nH, scale=scale, softcap=None, window=window, splits=splits)
        assert torch.equal(torch.isnan(out).all(1).cpu(), sees) and torch.equal(torch.isnan(out).any(1).cpu(), sees)
        for i in (at, at + 1, min(L, at + window) - 1):
            one = torch.empty_like(q[:1])
            ops.attention_f32(q[i:i + 1].contiguous(), kp, vp, one, ctx_of((i + 1,), (1,), pos[i:i + 1].contiguous(), seq[:1]), bt, num_heads=nH,
                              scale=scale, softcap=None, window=window, splits=splits)
            assert torch.isnan(one).all(), i


def test_attention_takes_rows_that_are_not_aligned():
    """The step's attention, as mixers call it, on queries and outputs at any address."""
    for lens, new in (((70, 33), (70, 33)), ((70, 33), (1, 1))):
        q, kp, vp, bt, pos, seq, ref, scale = attention_case("float32", 4, 2, 64, lens, new, 5.0, 20, seed=9)
        shifted = [torch.empty(q.numel() + 1, device=DEV)[1:].view_as(q) for _ in range(2)]
        shifted[0].copy_(q)
        for q_, out in ((q, shifted[1]), (shifted[0], torch.empty_like(q))):
            ops.attention(q_, kp, vp, out, ctx_of(lens, new, pos, seq), bt, num_heads=4, scale=scale, softcap=5.0, window=20, full_precision=True)
            close(out, ref, 1e-5)


def test_attention_refuses_what_is_outside_its_range():
    q, kp, vp, bt, pos, seq, _, scale = attention_case("float32", 4, 2, 32, (20,), (20,), None, None, seed=8)
    with pytest.raises(ops.HipLibraryError, match="outside"):
        ops.attention_f32(q, kp, vp, torch.empty_like(q), ctx_of((20,), (20,), pos, seq), bt, num_heads=4, scale=scale, softcap=None, window=None)
