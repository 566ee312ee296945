"""Tiled prompt attention at the ends of what it loads: last keys within a step of 32, head sizes that are padded, places of the
cache that are not written yet, with every term of the softmax and two page sizes, against plain attention in 64 bits."""
import types

import pytest
import torch

from alice_llm_amd.hip import ops
from test_gpu_kernels import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,d,dv", [(2, 1, 128, 128), (4, 4, 64, 40), (3, 1, 72, 256), (2, 1, 200, 64)])
@pytest.mark.parametrize("lens", [[257], [300, 1, 33], [64, 96, 128]])
@pytest.mark.parametrize("terms", [{}, dict(window=40), dict(window=70, keep_first=3), dict(chunk=100), dict(slopes=True, sink=True)])
@pytest.mark.parametrize("page", [64, 48])
def test_ends_against_plain_attention(H, G, d, dv, lens, page, terms):
    terms = dict(terms)
    gen = torch.Generator(device=DEV).manual_seed(d + sum(lens))
    T, B, width = sum(lens), len(lens), -(-max(lens) // page)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=gen).to(torch.bfloat16)                # noqa: E731
    kp, vp, q = rand(B * width, G, page, d), rand(B * width, G, page, dv), rand(T, H * d)
    if lens[-1] % page:                                      # places of the last page that are not written yet
        kp[-1, :, lens[-1] % page:], vp[-1, :, lens[-1] % page:] = float("nan"), float("nan")
    bt = torch.arange(B * width, dtype=torch.int32, device=DEV).view(B, width)
    starts = [sum(lens[:i]) for i in range(B + 1)]
    ctx = types.SimpleNamespace(positions=torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV), n_seqs=B,
                                cu_seqlens=torch.tensor(starts, dtype=torch.int32, device=DEV), max_position=max(lens) - 1)
    slopes = -torch.rand(H, device=DEV, generator=gen) / 20 if terms.pop("slopes", False) else None
    sink = torch.randn(H, device=DEV, generator=gen) if terms.pop("sink", False) else None
    window, chunk, keep = terms.get("window"), terms.get("chunk"), terms.get("keep_first", 0)
    out = torch.full((T, H * dv), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.attention_tiled(q, kp, vp, out, ctx, bt, num_heads=H, scale=d ** -0.5, bias_slopes=slopes, sink=sink, **terms)
    out = out.view(T, H, dv).double()
    for b, n in enumerate(lens):
        rows = lambda pool: pool[bt[b].long()].permute(1, 0, 2, 3).reshape(G, width * page, -1)[:, :n].double().repeat_interleave(H // G, 0)  # noqa: E731
        k, v = rows(kp), rows(vp)
        s = (q[starts[b]:starts[b + 1]].view(n, H, d).double().transpose(0, 1) @ k.transpose(1, 2).contiguous()) * d ** -0.5
        i, j = torch.arange(n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
        if slopes is not None:
            s = s + slopes.double()[:, None, None] * (j - i)
        lo = (i // chunk) * chunk if chunk else (i + 1 - window if window else torch.zeros_like(i))
        s = s.masked_fill((j > i) | ((j < lo) & (j >= keep)), float("-inf"))
        top = s.amax(-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink.double()[:, None, None])
        w = torch.exp(s - top)
        total = w.sum(-1, keepdim=True) + (torch.exp(sink.double()[:, None, None] - top) if sink is not None else 0)
        want = ((w / total) @ v).transpose(0, 1)
        # weights and output rounded to bfloat16: 8 significant bits, so half a unit is at most 2^-8 of the number; 32-bit sums
        # are far below
        bound = 2.0 ** -8 * (w / total @ v.abs()).transpose(0, 1) * 1.02 + 2.0 ** -8 * want.abs() * 1.02 + 1e-5
        assert bool(((out[starts[b]:starts[b + 1]] - want).abs() <= bound).all())
