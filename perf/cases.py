"""What is timed: steps of the library through its public entry points, over the sizes that its configurations,
tests and benchmark name.

Three paths: a step of whole prompts (`run_prompt_steps`, what the generation loop and the command line run first), a
step of one token for every sequence on top of its cached context (`Engine.step` with the ids on the device, what a
loop runs for every token after that) and the draw of the next tokens from logits (`Sampler`).  Outputs are the
float32 logits that a step returns, or the drawn ids.

Models: the Gemma 2 shapes 2B, 9B and 27B in bfloat16, the 2B shape on the true 32-bit path, and a Vifirax of six
layers (attention, state space, delta rule, each twice) whose feed-forwards are all dense: with random weights the
choice of experts is a near tie for some tokens of every step, and two correct implementations then give other logits.
Weights are random (bench.py's), tokens uniform, and the tokens of decode steps are given beforehand, as a trace
replay gives them, so that outputs do not hang on which of two near-equal logits was the larger.
"""
import math
import random

import torch

import alice_llm_amd as alice

DEVICE = "cuda"
FEEDS = 64                  # different tokens that decode steps of one state are fed, in turn
ROOM = {True: 4096, False: 1024}      # decode steps that a state's cache has room for: few sequences, many


def listed():
    return [
        # one user in a chat with a history: the smallest step there is, bound by latency and by reading the weights
        dict(name="decode-2b-b1", path="decode", model="2b", dtype="bfloat16", seqs=1, shortest=2048, longest=2048),
        # the headline of bench.py: eight users, equal histories
        dict(name="decode-2b-b8", path="decode", model="2b", dtype="bfloat16", seqs=8, shortest=2048, longest=2048),
        # a busy server: 64 users, histories from a greeting to a long chat
        dict(name="decode-2b-b64-ragged", path="decode", model="2b", dtype="bfloat16", seqs=64, shortest=64, longest=2048),
        # two long documents on the largest model, past the sliding window
        dict(name="decode-27b-b2-long", path="decode", model="27b", dtype="bfloat16", seqs=2, shortest=4400, longest=4700),
        # a question of a few lines: time to the first token
        dict(name="prompt-2b-117", path="prompt", model="2b", dtype="bfloat16", seqs=1, shortest=117, longest=117),
        # the headline prefill of bench.py
        dict(name="prompt-2b-2048", path="prompt", model="2b", dtype="bfloat16", seqs=1, shortest=2048, longest=2048),
        # a batch of unequal prompts at the 9B shape, in steps of the loop's token budget: the largest pass
        dict(name="prompts-9b-ragged", path="prompt", model="9b", dtype="bfloat16", seqs=16, shortest=64, longest=2048),
        # the 32-bit path, where logits are wanted without bfloat16's rounding: a prompt, and a few sequences' tokens
        dict(name="prompt-2b-f32-500", path="prompt", model="2b", dtype="float32", seqs=1, shortest=500, longest=500),
        dict(name="decode-2b-f32-b4", path="decode", model="2b", dtype="float32", seqs=4, shortest=300, longest=700),
        # attention beside fixed-size states: a long prompt, and a batch's tokens
        dict(name="prompt-vifirax-2048", path="prompt", model="vifirax", dtype="bfloat16", seqs=1, shortest=2048, longest=2048),
        dict(name="decode-vifirax-b8", path="decode", model="vifirax", dtype="bfloat16", seqs=8, shortest=500, longest=1500),
        # the draw behind a decode step of 64 sequences, with the usual cuts
        dict(name="sample-b64", path="sample", rows=64, vocab=256000, temperature=0.8, top_k=50, top_p=0.95),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["decode"] * 4 + ["prompt"] * 4 + ["sample"])
    if path == "sample":
        return dict(path=path, rows=_spread(rng, 1, 64), vocab=rng.choice([32768, 256000]), temperature=round(rng.uniform(0.3, 1.2), 2),
                    top_k=rng.choice([0, 20, 50, 200]), top_p=rng.choice([0.9, 0.95, 1.0]))
    model = rng.choice(["2b", "2b", "2b", "9b", "2b-f32", "vifirax", "vifirax"])
    dtype = "float32" if model == "2b-f32" else "bfloat16"
    if path == "decode":
        seqs = _spread(rng, 1, {"2b": 64, "9b": 24, "2b-f32": 8, "vifirax": 32}[model])
        most = {"2b": 60000, "9b": 16000, "2b-f32": 4000, "vifirax": 12000}[model] // seqs     # tokens of history in all
        longest = _spread(rng, 48, max(64, min(6000, most)))
    else:
        seqs = _spread(rng, 1, 8)
        most = {"2b": 20000, "9b": 12000, "2b-f32": 600, "vifirax": 12000}[model] // seqs
        longest = _spread(rng, 8, max(16, min(8000, most)))
    return dict(path=path, model=model.split("-")[0], dtype=dtype, seqs=seqs, shortest=rng.randint(max(1, longest // 16), longest), longest=longest)


# ---------------------------------------------------------------------------------- configurations and inputs

def config_of(case):
    """config.json of a case's model."""
    if case["model"] != "vifirax":
        raw = alice.preset(case["model"])
        raw["torch_dtype"] = case["dtype"]
        return raw
    width, ff, heads, kv, dim = 2048, 8192, 16, 4, 128            # bench.py's w2048
    dense = {"kind": "dense", "ff": ff}
    att = {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim, "scale": dim ** -0.5,
           "rot": {"base": 10000.0, "dims": dim // 2, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
    ssm = {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 1, "norm_groups": 1, "conv": 4}
    dlt = {"heads": heads, "kv_heads": heads, "dim": dim, "vdim": dim, "conv": 4, "decay_rank": dim, "gate_rank": dim}
    layers = [("attention", att), ("mamba2", ssm), ("channel_delta", dlt), ("attention", dict(att, kv_from=0)), ("mamba2", ssm),
              ("channel_delta", dlt)]
    return {"architecture": "Vifirax", "vocab": 32768, "width": width, "norm": {"eps": 1e-6}, "logit_scale": 0.5,
            "layers": [{"type": t, "mixer": m, "mlp": dense} for t, m in layers]}


def lengths(case):
    """Tokens of every sequence: the same for every seed."""
    rng = random.Random(case["seqs"] * 1000003 + case["shortest"] * 1009 + case["longest"])
    return [rng.randint(case["shortest"], case["longest"]) for _ in range(case["seqs"])]


def tokens_of(case, seed, vocab):
    """The prompts, and the tokens [FEEDS, seqs] that decode steps are fed."""
    gen = torch.Generator().manual_seed(seed + 1)
    prompts = [torch.randint(0, vocab, (n,), generator=gen).tolist() for n in lengths(case)]
    return prompts, torch.randint(0, vocab, (FEEDS, case["seqs"]), generator=gen, dtype=torch.int32)


def prepare(case, seed):
    if case["path"] == "sample":
        gen = torch.Generator(device=DEVICE).manual_seed(seed)
        logits = torch.randn(case["rows"], case["vocab"], device=DEVICE, generator=gen).mul_(4.0)
        logits = torch.tanh(logits / 30.0).mul_(30.0)             # what capped logits look like
        return dict(path="sample", logits=logits, requests=list(range(case["rows"])), draws=[7] * case["rows"],
                    sampler=alice.Sampler(case["temperature"], case["top_k"], case["top_p"], seed=seed))
    model = alice.Model.random(config_of(case), seed=seed, dtype=case["dtype"], fast=True)
    prompts, feeds = tokens_of(case, seed, model.lm.plan.vocab_size)
    lens = lengths(case)
    state = dict(path=case["path"], model=model, prompts=prompts)
    if case["path"] == "prompt":
        state["engine"] = model.engine(seq_lens=lens, max_seqs=len(lens))
        return state
    room = min(ROOM[case["seqs"] <= 8], model.lm.plan.max_positions - max(lens))
    state.update(engine=model.engine(seq_lens=[n + room for n in lens], max_seqs=len(lens)), room=room,
                 feeds=list(feeds.to(DEVICE).unbind(0)), slots=None)
    _begin(state)
    return state


def _begin(state):
    """The sequences' prompts and first decode step: a program that decodes has these behind it."""
    engine = state["engine"]
    if state["slots"] is not None:
        engine.close(state["slots"])
    state["slots"] = engine.open(len(state["prompts"]))
    alice.run_prompt_steps(engine, state["slots"], state["prompts"])
    engine.step(state["slots"], state["feeds"][0], "last")
    state["at"] = 1


def run(state):
    if state["path"] == "sample":
        return state["sampler"](state["logits"], state["requests"], state["draws"])
    engine = state["engine"]
    if state["path"] == "prompt":
        slots = engine.open(len(state["prompts"]))
        logits = alice.run_prompt_steps(engine, slots, state["prompts"])
        engine.close(slots)
        return logits
    if state["at"] >= state["room"]:
        _begin(state)                                             # the sequences ended: the next ones
    logits = engine.step(state["slots"], state["feeds"][state["at"] % FEEDS], "last")
    state["at"] += 1
    return logits


# ---------------------------------------------------------------------------------- the work of a pass

def _shapes(raw):
    """(matrix weights without the embedding, embedding rows, their width)."""
    n = sum(math.prod(shape) for name, shape, _, _ in tensors_of(raw) if len(shape) == 2)
    vocab, width = (raw["vocab"], raw["width"]) if "vocab" in raw else (raw["vocab_size"], raw["hidden_size"])
    return n - vocab * width, vocab, width


def work(case):
    if case["path"] == "sample":
        return {"bytes": 4 * case["rows"] * case["vocab"], "flops": 4 * case["rows"] * case["vocab"]}
    raw, elem = config_of(case), 2 if case["dtype"] == "bfloat16" else 4
    matrices, vocab, width = _shapes(raw)
    lens = lengths(case)
    pairs = []                                                    # (query, key) pairs and key rows of each attention layer
    if case["model"] == "vifirax":
        heads, kv, dim = 16, 4, 128
        windows, own = [None, None], 1                            # the second reads the first one's keys
        state = 2 * (64 * 128 * 64 + 16 * 128 * 128)              # numbers of state a sequence
        scan = 2 * 6 * (64 * 128 * 64) + 2 * 8 * (16 * 128 * 128)  # operations on it a token
    else:
        heads, kv, dim = raw["num_attention_heads"], raw["num_key_value_heads"], raw["head_dim"]
        windows, state, scan = [raw["sliding_window"] if i % 2 == 0 else None for i in range(raw["num_hidden_layers"])], 0, 0
        own = len(windows)
    keys_read = 0
    for w in windows:
        for n in lens:
            if case["path"] == "decode":
                seen = n + 2 if w is None else min(n + 2, w)
                pairs.append(seen)
                keys_read += seen
            else:
                pairs.append(n * (n + 1) // 2 if w is None or w >= n else w * (w + 1) // 2 + (n - w) * w)
    new = len(lens) if case["path"] == "decode" else sum(lens)
    flops = 2 * new * matrices + 2 * len(lens) * vocab * width + 4 * heads * dim * sum(pairs) + new * scan
    row = 2 * kv * dim * elem
    nbytes = (matrices + vocab * width) * elem + keys_read * row + new * own * row + len(lens) * vocab * 4
    nbytes += len(lens) * state * 4 * (2 if case["path"] == "decode" else 1)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["path"] == "sample":
        return "exact"
    # measured against 64 bits: 0.6 to 1.3 % in bfloat16, 2e-6 to 5e-6 in 32-bit
    return {"rel": 0.03, "max": 0.3} if case["dtype"] == "bfloat16" else {"rel": 2e-5, "max": 4e-4}


# ---------------------------------------------------------------------------------- the same in 64 bits

F64 = torch.float64


def tensors_of(raw):
    """(name, shape, mean, deviation) of every tensor, in the order in which random weights are drawn."""
    if raw.get("architecture") == "Vifirax":
        V, W = raw["vocab"], raw["width"]
        yield "embed", (V, W), 0.0, 0.02
        for i, layer in enumerate(raw["layers"]):
            m, ff, p = layer["mixer"], layer["mlp"]["ff"], f"l{i}."
            H, P = m["heads"], m["vdim"]
            if layer["type"] == "attention":
                Q, K, own = H * m["dim"], m["kv_heads"] * m["dim"], "kv_from" not in m
                names = [("q", (Q, W), 0.02)] + ([("k", (K, W), 0.02), ("v", (K, W), 0.02)] if own else [])
                names += [("o", (W, Q), 0.02), ("g", (H, W), 0.02), ("q.b", (Q,), 0.1)]
                names += [("k.b", (K,), 0.1), ("v.b", (K,), 0.1)] if own else []
                names += [("q.norm", (Q,), 0.3)] + ([("k.norm", (K,), 0.3)] if own else []) + [("o.b", (W,), 0.1)]
            elif layer["type"] == "mamba2":
                inner, ch = H * P, H * P + 2 * m["groups"] * m["state"]
                names = [("in", (inner + ch + H, W), 0.02), ("conv", (ch, m["conv"]), 0.3), ("conv.b", (ch,), 0.1), ("dt_bias", (H,), 0.5),
                         ("A_log", (H,), 0.5), ("D", (H,), 0.5), ("norm", (inner,), 0.3), ("o", (W, inner), 0.02)]
            else:
                Q, ra, rg = H * m["dim"], m["decay_rank"], m["gate_rank"]
                names = [(n + s, shape, std) for n in "qkv" for s, shape, std in (("", (Q, W), 0.02), (".conv", (Q, m["conv"]), 0.3))]
                names += [("b", (H, W), 0.02), ("A_log", (H,), 0.5), ("norm", (P,), 0.3), ("a1", (ra, W), 0.02), ("a2", (Q, ra), 0.3),
                          ("dt_bias", (Q,), 0.5), ("g1", (rg, W), 0.02), ("g2", (Q, rg), 0.3), ("o", (W, Q), 0.02)]
            for n, shape, std in names:
                yield p + "mix." + n, shape, 0.0, std
            for n, shape, std in (("mlp.gate", (ff, W), 0.02), ("mlp.up", (ff, W), 0.02), ("mlp.down", (W, ff), 0.02), ("norm1", (W,), 0.1),
                                  ("norm2", (W,), 0.1)):
                yield p + n, shape, 0.0, std
        yield "final.norm", (W,), 0.0, 0.1
        return
    W, ff, d = raw["hidden_size"], raw["intermediate_size"], raw["head_dim"]
    Q, K = raw["num_attention_heads"] * d, raw["num_key_value_heads"] * d
    yield "embed", (raw["vocab_size"], W), 0.0, 0.02
    for i in range(raw["num_hidden_layers"]):
        for n, shape, std in (("q", (Q, W), 0.02), ("k", (K, W), 0.02), ("v", (K, W), 0.02), ("o", (W, Q), 0.02), ("gate", (ff, W), 0.02),
                              ("up", (ff, W), 0.02), ("down", (W, ff), 0.02), ("n1", (W,), 0.1), ("n1b", (W,), 0.1), ("n2", (W,), 0.1),
                              ("n2b", (W,), 0.1)):
            yield f"l{i}.{n}", shape, 0.0, std
    yield "final", (W,), 0.0, 0.1


class Weights:
    """The tensors one after another, as Model.random(fast=True) draws them, each kept until its layer is done."""

    def __init__(self, raw, seed):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)
        self.specs = tensors_of(raw)
        self.dtype = torch.float32 if raw.get("torch_dtype") == "float32" else torch.bfloat16
        self.kept = {}

    def get(self, name):
        while name not in self.kept:
            n, shape, mean, std = next(self.specs)
            t = torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(mean, std, generator=self.gen)
            self.kept[n] = t.to(self.dtype)
        return self.kept[name].to(F64)

    def rows(self, name, idx):
        if name not in self.kept:
            self.get(name)
        return self.kept[name][idx].to(F64)

    def drop(self, prefix):
        for n in [n for n in self.kept if n.startswith(prefix)]:
            del self.kept[n]


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _by_rows(f, x, step=8192):
    return torch.cat([f(part) for part in x.split(step)])


def _turn(x, positions, freqs, m=1.0):
    """Dimension i < R/2 of every head turned with i + R/2; x [T, heads, d], R = 2 len(freqs)."""
    half = freqs.numel()
    ang = positions.to(F64)[:, None] * freqs[None]
    c, s = (torch.cos(ang) * m)[:, None], (torch.sin(ang) * m)[:, None]
    out = x.clone()
    u, v = x[..., :half], x[..., half:2 * half]
    out[..., :half], out[..., half:2 * half] = u * c - v * s, v * c + u * s
    return out


def _attend(q, k, v, scale, cap, window, one_more):
    """q [T, H, d], k and v [T, G, d] of one sequence; rows of queries at a time."""
    T, H, d = q.shape
    G = k.shape[1]
    q = q.view(T, G, H // G, d)
    step = max(1, int(2e8 // (H * T)))
    at, out = torch.arange(T, device=q.device), torch.empty_like(q)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    for i in range(0, T, step):
        rows = at[i:i + step]
        n = rows.numel()
        hi = i + n
        lo = 0 if window is None else max(0, i + 1 - window)
        s = torch.matmul(q[i:hi].permute(1, 0, 2, 3).reshape(G, n * (H // G), d), kt[:, :, lo:hi].contiguous()).mul_(scale)
        if cap:
            s = s.div_(cap).tanh_().mul_(cap)
        back = rows[:, None] - at[None, lo:hi]
        hidden = (back < 0) if window is None else (back < 0) | (back >= window)
        s = s.view(G, n, H // G, hi - lo).masked_fill_(hidden[None, :, None], -math.inf)
        top = s.amax(-1, keepdim=True)
        if one_more:
            top = top.clamp(min=0.0)
        s = s.sub_(top).exp_()
        total = s.sum(-1, keepdim=True)
        s = s.div_(total + torch.exp(-top) if one_more else total)
        out[i:hi] = torch.matmul(s.view(G, n * (H // G), hi - lo), vt[:, lo:hi]).view(G, n, H // G, -1).permute(1, 0, 2, 3)
    return out.reshape(T, H * d)


def _gemma(raw, w, ids, lens):
    eps, d = raw["rms_norm_eps"], raw["head_dim"]
    H, G = raw["num_attention_heads"], raw["num_key_value_heads"]
    norm = lambda x, n: _unit(x, eps) * (1.0 + w.get(n))                                       # noqa: E731
    positions = torch.cat([torch.arange(n, device=DEVICE) for n in lens])
    freqs = raw["rope_theta"] ** (-torch.arange(0, d, 2, dtype=F64, device=DEVICE) / d)
    x = w.rows("embed", ids) * float(torch.tensor(float(raw["hidden_size"])).sqrt())
    for i in range(raw["num_hidden_layers"]):
        p, window = f"l{i}.", raw["sliding_window"] if i % 2 == 0 else None
        w.get(p + "n2b")
        h = norm(x, p + "n1")
        q, k = ((h @ w.get(p + n).T).view(len(ids), -1, d) for n in "qk")
        v = (h @ w.get(p + "v").T).view(len(ids), G, d)
        q, k = _turn(q, positions, freqs), _turn(k, positions, freqs)
        scale, cap = raw["query_pre_attn_scalar"] ** -0.5, raw["attn_logit_softcapping"]
        a = torch.cat([_attend(*t, scale, cap, window, False) for t in zip(q.split(lens), k.split(lens), v.split(lens))])
        del q, k, v
        x = x + norm(a @ w.get(p + "o").T, p + "n1b")
        gate, up, down = (w.get(p + n).T for n in ("gate", "up", "down"))
        gelu = lambda z: torch.nn.functional.gelu(z, approximate="tanh")                       # noqa: E731
        x = x + norm(_by_rows(lambda r: (gelu(r @ gate) * (r @ up)) @ down, norm(x, p + "n2")), p + "n2b")
        w.drop(p)
    last = torch.tensor(lens, device=DEVICE).cumsum(0) - 1
    z, cap = norm(x[last], "final") @ w.get("embed").T, raw["final_logit_softcapping"]
    return cap * torch.tanh(z / cap)


def _stretched(dims, base, sc):
    i = torch.arange(dims // 2, dtype=F64, device=DEVICE)
    f = base ** (-2.0 * i / dims)
    where = lambda turns: dims * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))   # noqa: E731
    lo, hi = max(math.floor(where(sc["fast"])), 0), min(math.ceil(where(sc["slow"])), dims - 1)
    r = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / sc["factor"] * r + f * (1 - r), 0.1 * math.log(sc["factor"]) + 1.0


def _conv(x, weight, bias, lens):
    """A causal convolution a channel over each sequence, then silu."""
    taps, out = weight.shape[1], []
    for part in x.split(lens):
        padded = torch.cat([part.new_zeros(taps - 1, part.shape[1]), part])
        out.append(sum(padded[j:j + part.shape[0]] * weight[:, j] for j in range(taps)))
    y = torch.cat(out) if bias is None else torch.cat(out) + bias
    return y * torch.sigmoid(y)


def _vifirax(raw, w, ids, lens):
    eps, T = raw["norm"]["eps"], len(ids)
    silu = torch.nn.functional.silu
    positions = torch.cat([torch.arange(n, device=DEVICE) for n in lens])
    norm = lambda x, n: _unit(x, eps) * (1.0 + w.get(n))                                       # noqa: E731
    x, made = w.rows("embed", ids), {}
    for i, layer in enumerate(raw["layers"]):
        p, m = f"l{i}.mix.", layer["mixer"]
        H, P = m["heads"], m["vdim"]
        w.get(f"l{i}.norm2")
        lin = lambda n, h=x: h @ w.get(p + n).T                                                # noqa: E731
        if layer["type"] == "attention":
            d, rot = m["dim"], m["rot"]
            turn = lambda t: _turn(t, positions, *_stretched(rot["dims"], rot["base"], rot["scaling"]))   # noqa: E731
            if "kv_from" not in m:
                k = turn((_unit(lin("k") + w.get(p + "k.b"), eps) * w.get(p + "k.norm")).view(T, -1, d))
                made[i] = k, (lin("v") + w.get(p + "v.b")).view(T, -1, d)
            k, v = made[m.get("kv_from", i)]
            q = turn((_unit(lin("q") + w.get(p + "q.b"), eps) * w.get(p + "q.norm")).view(T, H, d))
            a = torch.cat([_attend(*t, m["scale"], None, None, True) for t in zip(q.split(lens), k.split(lens), v.split(lens))])
            y = (a.view(T, H, d) * torch.sigmoid(lin("g"))[..., None]).reshape(T, H * d) @ w.get(p + "o").T + w.get(p + "o.b")
        elif layer["type"] == "mamba2":
            N, inner = m["state"], H * P
            z, u, dt = lin("in").split([inner, inner + 2 * N, H], dim=1)
            u, B, C = _conv(u, w.get(p + "conv"), w.get(p + "conv.b"), lens).split([inner, N, N], dim=1)
            u, dt = u.reshape(T, H, P), torch.nn.functional.softplus(dt + w.get(p + "dt_bias"))
            keep, o = torch.exp(-torch.exp(w.get(p + "A_log")) * dt)[:, :, None, None], torch.empty_like(u)
            du, D, t = dt[:, :, None] * u, w.get(p + "D")[:, None], 0
            for n in lens:
                S = u.new_zeros(H, N, P)
                for t in range(t, t + n):
                    S = torch.addcmul(keep[t] * S, B[t][None, :, None], du[t][:, None, :])
                    o[t] = torch.matmul(C[t], S)
                t += 1
            y = _unit((o + D * u).reshape(T, inner) * silu(z), eps) * w.get(p + "norm") @ w.get(p + "o").T
        else:
            d = m["dim"]
            q, k, v = (_conv(lin(n), w.get(p + n + ".conv"), None, lens).view(T, H, -1) for n in "qkv")
            q, k = (a / torch.sqrt((a * a).sum(-1, keepdim=True) + 1e-6) for a in (q, k))
            q, beta = q * d ** -0.5, torch.sigmoid(lin("b"))
            low = torch.nn.functional.softplus(lin("a1") @ w.get(p + "a2").T + w.get(p + "dt_bias")).view(T, H, d)
            g, o, t = torch.exp(-torch.exp(w.get(p + "A_log"))[:, None] * low), torch.empty_like(v), 0
            bk = beta[..., None] * k
            for n in lens:
                S = v.new_zeros(H, d, P)
                for t in range(t, t + n):
                    S = g[t][..., None] * S
                    S = torch.baddbmm(S, bk[t][..., None], v[t][:, None] - torch.bmm(k[t][:, None], S))
                    o[t] = torch.bmm(q[t][:, None], S)[:, 0]
                t += 1
            gate = torch.sigmoid(lin("g1") @ w.get(p + "g2").T).view(T, H, P)
            y = (_unit(o, eps) * w.get(p + "norm") * gate).reshape(T, H * P) @ w.get(p + "o").T
        p = f"l{i}."
        x = x + norm(y, p + "norm1")
        gate, up, down = (w.get(p + "mlp." + n).T for n in ("gate", "up", "down"))
        x = x + norm(_by_rows(lambda r: (silu(r @ gate) * (r @ up)) @ down, x), p + "norm2")
        w.drop(p)
    last = torch.tensor(lens, device=DEVICE).cumsum(0) - 1
    return norm(x[last], "final.norm") @ w.get("embed").T * raw["logit_scale"]


def exact(case, seed):
    """A step's logits in 64 bits: whole sequences, no cache."""
    if case["path"] == "sample":
        return None                                               # whole numbers
    raw = config_of(case)
    prompts, feeds = tokens_of(case, seed, raw.get("vocab_size") or raw["vocab"])
    if case["path"] == "decode":                                  # the two tokens that prepare and the first pass feed
        prompts = [p + feeds[:2, i].tolist() for i, p in enumerate(prompts)]
    ids = torch.tensor([t for p in prompts for t in p], device=DEVICE)
    forward = _vifirax if raw.get("architecture") == "Vifirax" else _gemma
    return forward(raw, Weights(raw, seed), ids, [len(p) for p in prompts])
