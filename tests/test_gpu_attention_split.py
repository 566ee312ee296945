"""Single-token attention with the keys split over blocks: rows of every number of lanes, groups of every register form, runs
around 32 and 256 keys, against plain attention in 64 bits."""
import pytest
import torch

from alice_llm_amd.hip import ops
from test_gpu_kernels import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,d,dv", [(1, 1, 8, 8), (2, 2, 16, 24), (6, 2, 32, 64), (4, 1, 64, 40), (8, 1, 96, 128), (16, 1, 128, 128), (10, 2, 256, 16),
                                      (4, 1, 136, 256), (3, 1, 40, 104), (16, 1, 256, 256)])
def test_against_plain_attention(dtype, H, G, d, dv):
    gen = torch.Generator(device=DEV).manual_seed(H * d + dv)
    lens, page = [1, 31, 33, 255, 256, 257, 520], 64
    T, most = len(lens), max(lens)
    width = -(-most // page)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=gen).to(dtype)                        # noqa: E731
    kp, vp, q = rand(T * width, G, page, d), rand(T * width, G, page, dv), rand(T, H * d)
    bt = torch.randperm(T * width, device=DEV, generator=gen).to(torch.int32).view(T, width)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)                                        # noqa: E731
    pos, seq, scale = i32([n - 1 for n in lens]), i32(list(range(T))), d ** -0.5
    out, per = torch.full((T, H * dv), float("nan"), dtype=dtype, device=DEV), torch.full((T, H, G, dv), float("nan"), device=DEV)
    common = dict(num_heads=H, scale=scale, max_position=most - 1, max_keys=most)
    ops.attention_split(q, kp, vp, out, pos, seq, bt, **common)
    ops.attention_split(q, kp, vp, None, pos, seq, bt, per_value_head=per, **common)
    for t, n in enumerate(lens):
        rows = lambda pool: pool[bt[t].long()].permute(1, 0, 2, 3).reshape(G, width * page, -1)[:, :n].double()     # noqa: E731
        k, v = rows(kp).repeat_interleave(H // G, 0), rows(vp)
        qt = q[t].view(H, 1, d).double()
        w = torch.softmax((qt * k).sum(-1) * scale, -1)                                                  # [H, n]
        want = (w[:, None, :, None] * v[None]).sum(2)                                                    # [H, G, dv]
        # 32-bit sums of d products, of n weights and of n weighted values, and exponents of up to 16 in 32 bits
        e = 2.0 ** -24
        score = (d + 2) * e * float((qt * k).abs().sum(-1).max()) * scale
        bound = float(v.abs().max()) * (2 * score + (2 * n + 64) * e)
        assert float((per[t].double() - want).abs().max()) <= bound
        own = want[torch.arange(H), torch.arange(H) // (H // G)]
        err = (out[t].view(H, dv).double() - own).abs()
        assert bool((err <= bound + (2.0 ** -8 * own.abs() if dtype == torch.bfloat16 else 0)).all())
