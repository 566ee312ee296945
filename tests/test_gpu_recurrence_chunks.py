"""The matrix recurrences by chunks of 16 tokens against the plain token-by-token scans in 64 bits."""
from types import SimpleNamespace

import pytest
import torch

from alice_llm_amd.hip import ops
from plain import vifirax_plain as P
from test_gpu_vifirax import DEV, _Ctx, max_err, rnd

pytestmark = pytest.mark.gpu

# two steps over three slots: pieces that end within a chunk, at its end and one token behind it, and single tokens
STEPS = [([33, 16, 1, 47], [2, 0, 5, 3]), ([1, 17, 15, 64], [5, 0, 3, 2])]


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("strength", [0.05, 1.0, 30.0])
@pytest.mark.parametrize("H,G,d,dv", [(4, 2, 8, 16), (3, 3, 12, 20), (2, 1, 64, 128), (1, 1, 136, 24), (2, 2, 200, 7), (70, 1, 16, 8), (2, 2, 256, 17)])
def test_chunks_over_pieces_and_slots(delta, strength, H, G, d, dv):
    """`strength`: the size of the decays' logarithms a token, from slow ones to such that a chunk's product underflows."""
    per, total = H // G, {slot: 0 for _, slots in STEPS for slot in slots}
    S = torch.full((6, H, d, dv), 3.0, device=DEV)
    S[list(total)] = 0.0
    state = {slot: None for slot in total}
    skip = None if delta else rnd(H, seed=3)
    for step, (lens, slots) in enumerate(STEPS):
        T = sum(lens)
        q, k, v = rnd(T, G * d + 4, seed=20 + step), rnd(T, G * d, seed=30 + step), rnd(T, H * dv, seed=40 + step)
        if delta:
            q[:, :G * d] = P.unit_vectors(q[:, :G * d].view(T, G, d)).reshape(T, G * d)
            k = P.unit_vectors(k.view(T, G, d)).reshape(T, G * d)
        log = -strength * rnd(T, H * d if delta else H, seed=50 + step).abs()
        b = torch.sigmoid(rnd(T, H, seed=60 + step)) * (1.0 if delta else 2.0)
        out = torch.full((T, H * dv), float("nan"), device=DEV)
        ops.recurrence_chunks(q.to(DEV), 0, k.to(DEV), 0, v.to(DEV), 0, log.to(DEV), b.to(DEV), None if skip is None else skip.to(DEV),
                              out, _Ctx(lens, slots), S, heads=H, qk_heads=G, head_dim=d, value_head_dim=dv, delta=delta)
        at = 0
        for n, slot in zip(lens, slots):
            r = slice(at, at + n)
            qh, kh = (x[r, :G * d].double().view(n, G, d).repeat_interleave(per, dim=1) for x in (q, k))
            vh, decay = v[r].double().view(n, H, dv), torch.exp(log[r].double())
            if delta:
                ref, state[slot] = P.delta_rule_scan(qh, kh, vh, decay.view(n, H, d), b[r].double(), state[slot])
            else:
                # the plain scan takes step sizes and rates of one; the write's factor is given by scaling the values
                dt = -log[r].double()
                u = vh * (b[r].double() / dt)[:, :, None]
                ref, state[slot] = P.state_space_scan(u, kh, qh, dt, torch.zeros(H).double(), torch.zeros(H).double(), state[slot])
                ref = ref + skip.double()[None, :, None] * vh
            # sums over a few hundred terms of order one and their products with queries of the same size
            assert max_err(out[r], ref.reshape(n, H * dv)) < 2e-5 * max(1.0, float(ref.abs().max())), (step, slot)
            assert max_err(S[slot], state[slot]) < 2e-5 * max(1.0, float(state[slot].abs().max())), (step, slot)
            at += n
    others = [i for i in range(6) if i not in total]
    assert float((S[others] - 3.0).abs().max()) == 0.0                  # rows of other slots are untouched


def test_sizes_outside_the_range_stay_with_the_token_by_token_kernel():
    ctx = SimpleNamespace(max_new=ops.RECURRENCE_CHUNKS_FROM, n_seqs=1)
    kw = dict(heads=2, qk_heads=2, value_head_dim=16, delta=True)
    assert ops.recurrence_by_chunks(ctx, 64, 0, head_dim=16, **kw)
    assert not ops.recurrence_by_chunks(ctx, 64, 0, head_dim=18, **kw) and not ops.recurrence_by_chunks(ctx, 63, 0, head_dim=16, **kw)
    assert not ops.recurrence_by_chunks(SimpleNamespace(max_new=ops.RECURRENCE_CHUNKS_FROM - 1, n_seqs=1), 64, 0, head_dim=16, **kw)
    many = SimpleNamespace(max_new=400, n_seqs=ops.DELTA_CHUNKS_WAVES // 2 + 1)
    assert not ops.recurrence_by_chunks(many, 64, 0, head_dim=16, **kw)
    assert ops.recurrence_by_chunks(many, 64, 0, head_dim=16, **dict(kw, delta=False))


@pytest.mark.parametrize("delta", [False, True])
def test_both_block_sizes_give_the_same(delta):
    """Key sizes of 65 to 128 take eight waves a block, or four where there are 512 blocks and more: the same pieces alone
    and 64 times over."""
    H, d, dv, n = 2, 96, 64, 35
    q, k, v = (rnd(n, H * w, seed=i).to(DEV) for i, w in ((1, d), (2, d), (3, dv)))
    log, b = -rnd(n, H * d if delta else H, seed=4).abs().to(DEV), torch.sigmoid(rnd(n, H, seed=5)).to(DEV)
    outs = []
    for copies in (1, 64):
        S, out = torch.zeros(copies, H, d, dv, device=DEV), torch.empty(copies * n, H * dv, device=DEV)
        many = [x.repeat(copies, 1) for x in (q, k, v, log, b)]
        ops.recurrence_chunks(many[0], 0, many[1], 0, many[2], 0, many[3], many[4], None, out, _Ctx([n] * copies, list(range(copies))), S,
                              heads=H, qk_heads=H, head_dim=d, value_head_dim=dv, delta=delta)
        outs.append((out.view(copies, n, H * dv), S))
    (a, sa), (c, sc) = outs
    assert (c - a).abs().max() < 1e-5 * a.abs().max() and (sc - sa).abs().max() < 1e-5 * sa.abs().max()


def scan64(q, k, v, decay, b, H, delta):
    """Token by token in 64 bits: q, k [T, H, d], v [T, H, dv], decay [T, H, d or 1], b [T, H] -> [T, H dv], the state."""
    q, k, v, decay, b = (x.double() for x in (q, k, v, decay, b))
    S, out = q.new_zeros(H, q.shape[2], v.shape[2]), []
    for t in range(len(q)):
        S = decay[t][:, :, None] * S
        u = v[t] - (torch.matmul(k[t][:, None], S)[:, 0] if delta else 0.0)
        S = S + k[t][:, :, None] * (b[t][:, None] * u)[:, None]
        out.append(torch.matmul(q[t][:, None], S).reshape(-1))
    return torch.stack(out), S


def case(T, H, d, dv, delta, strength, seed=0):
    q, k, v = (rnd(T, H * w, seed=seed + i).to(DEV) for i, w in ((1, d), (2, d), (3, dv)))
    if delta:
        q, k = ((x.view(T, H, d) / x.view(T, H, d).norm(dim=-1, keepdim=True)).reshape(T, -1) for x in (q, k))
    log, b = -strength * rnd(T, H * d if delta else H, seed=seed + 4).abs().to(DEV), torch.sigmoid(rnd(T, H, seed=seed + 5)).to(DEV)
    return q, k, v, log, b


def both_ways(T, H, d, dv, delta, q, k, v, log, b):
    """(by chunks, token by token): out and state of each."""
    kw, res = dict(heads=H, qk_heads=H, head_dim=d, value_head_dim=dv, delta=delta), []
    for chunks in (True, False):
        S, out = torch.zeros(1, H, d, dv, device=DEV), torch.empty(T, H * dv, device=DEV)
        if chunks:
            ops.recurrence_chunks(q, 0, k, 0, v, 0, log, b, None, out, _Ctx([T], [0]), S, **kw)
        else:
            ops.matrix_recurrence(q, 0, k, 0, v, 0, torch.exp(log), b, None, out, _Ctx([T], [0]), S, decay_per_channel=delta, **kw)
        res.append((out, S[0]))
    return res


@pytest.mark.parametrize("delta,H,d,dv", [(False, 64, 128, 64), (True, 16, 128, 128), (True, 8, 64, 64), (False, 8, 256, 64)])
@pytest.mark.parametrize("strength", [0.01, 0.1, 1.0, 5.0])
def test_chunks_are_as_near_to_64_bits_as_token_by_token(delta, H, d, dv, strength):
    """The 2-norms of the errors over 300 tokens: 0.6 to 1.25 of the token-by-token kernel's, which adds up a product with a key in as
    many sums as it has lanes (1.7 to 3.2 with one sum over a key)."""
    T = 300
    args = case(T, H, d, dv, delta, strength)
    q, k, v, log, b = args
    ref, S = scan64(q.view(T, H, d), k.view(T, H, d), v.view(T, H, dv), torch.exp(log.double()).view(T, H, -1), b, H, delta)
    (a, sa), (c, sc) = both_ways(T, H, d, dv, delta, *args)
    assert (a - ref).norm() < 1.4 * (c - ref).norm() and (sa - S).norm() < 1.4 * (sc - S).norm()


@pytest.mark.parametrize("delta", [False, True])
def test_a_decay_of_zero_forgets(delta):
    """Logarithms of minus infinity, and ones far below what 32 bits hold: the state before is gone, nothing else."""
    T, H, d, dv = 70, 2, 12, 20
    q, k, v, log, b = case(T, H, d, dv, delta, 0.3)
    log[21], log[40], log[41] = -float("inf"), -3e38, -2e5
    if delta:
        log[52, 5] = -float("inf")
    ref, S = scan64(q.view(T, H, d), k.view(T, H, d), v.view(T, H, dv), torch.exp(log.double()).view(T, H, -1), b, H, delta)
    for out, state in both_ways(T, H, d, dv, delta, q, k, v, log, b):
        assert (out - ref).abs().max() < 2e-5 and (state - S).abs().max() < 2e-5


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("what", ["q", "k", "v", "log", "b"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("d,dv", [(12, 20), (128, 64), (256, 16)])
def test_what_is_no_finite_number_reaches_no_earlier_token(delta, what, value, d, dv):
    """One such number in the first head at a chunk's first, middle and last token and at the last one of all: the outputs that it
    reaches are those of the scan in 64 bits, and the others are what they are without it."""
    if what == "log" and value == float("inf"):
        value = -value                                                  # (no decay is above one; this one is zero: nothing is lost)
    T, H = 70, 2
    for at in (16, 21, 31, 69):
        args = dict(zip(("q", "k", "v", "log", "b"), case(T, H, d, dv, delta, 0.3, seed=at)))
        args[what][at, 0 if what == "b" or what == "log" and not delta else 3] = value
        q, k, v, log, b = args.values()
        ref, S = scan64(q.view(T, H, d), k.view(T, H, d), v.view(T, H, dv), torch.exp(log.double()).view(T, H, -1), b, H, delta)
        fine, there = torch.isfinite(ref), torch.isfinite(S)
        assert fine[:at].all() and fine[:, dv:].all()
        out, state = both_ways(T, H, d, dv, delta, q, k, v, log, b)[0]
        assert torch.equal(torch.isfinite(out), fine) and torch.equal(torch.isfinite(state), there), at
        assert (out - ref)[fine].abs().max() < 2e-5 * max(1.0, float(ref[fine].abs().max()))
        assert (state - S)[there].abs().max() < 2e-5 * max(1.0, float(S[there].abs().max()))


@pytest.mark.parametrize("delta,H,d,dv,lens", [(True, 512, 256, 16, [300]), (True, 300, 256, 20, [40, 230, 7, 129]), (False, 4096, 64, 4, [1500]),
                                              (False, 3000, 64, 4, [900, 33, 600])])
def test_a_step_beyond_the_workspace_goes_in_runs(delta, H, d, dv, lens):
    """More chunks than 256 MB hold: in runs, with the token-by-token kernel's result, and from no more memory."""
    T, G = sum(lens), 1
    per = ops.library().alice_recurrence_chunks_workspace(16, 1, H, G, d, dv, int(delta)) // 2
    need = ops.library().alice_recurrence_chunks_workspace(T, len(lens), H, G, d, dv, int(delta))
    assert need <= 1 << 26 and need < per * sum(-(-n // 16) for n in lens)
    q, k, v = (rnd(T, w, seed=i).to(DEV) for i, w in ((1, G * d), (2, G * d), (3, H * dv)))
    q, k = (x / x.norm(dim=1, keepdim=True) for x in (q, k))
    log, b = -0.3 * rnd(T, H * d if delta else H, seed=4).abs().to(DEV), torch.sigmoid(rnd(T, H, seed=5)).to(DEV)
    ctx, kw, res = _Ctx(lens, list(range(len(lens)))), dict(heads=H, qk_heads=G, head_dim=d, value_head_dim=dv, delta=delta), []
    for chunks in (True, False):
        S, out = torch.zeros(len(lens), H, d, dv, device=DEV), torch.full((T, H * dv), float("nan"), device=DEV)
        if chunks:
            ctx.max_new = max(lens)
            ops.recurrence_chunks(q, 0, k, 0, v, 0, log, b, None, out, ctx, S, **kw)
        else:
            ops.matrix_recurrence(q, 0, k, 0, v, 0, torch.exp(log), b, None, out, ctx, S, decay_per_channel=delta, **kw)
        res.append((out, S))
    for x, y in zip(*res):
        assert (x - y).abs().max() < 2e-5 * max(1.0, float(y.abs().max()))
