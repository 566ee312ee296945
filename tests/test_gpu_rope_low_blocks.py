"""The fused q, k, v product in blocks of 32 tokens (few tokens, no more blocks than the chip has places): the same bits as the tiled
product and the rotation one after the other."""
import pytest
import torch

from alice_llm_amd.hip import ops
from test_gpu_kernels import acts_to_fragments, pair_order, paged, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"


# heads and widths of the 2B and the 9B shape; rows that are no multiple of a block's 64, an inner dimension of a partial stage;
# tokens: first and last of the rule's range, a token tile missing from the last block, a single token in it, a partial tile
@pytest.mark.parametrize("nH,nKV,d,K,tokens", [(8, 4, 256, 2304, (65, 80, 97, 117, 128)), (16, 8, 256, 3584, (33, 47, 64)), (5, 1, 96, 1056, (66, 127, 200, 700)),
                                               (1, 1, 32, 32, (65, 1024))])
@pytest.mark.parametrize("layout", [0, 1])
def test_blocks_of_32_tokens(nH, nKV, d, K, tokens, layout):
    N = (nH + 2 * nKV) * d
    w = ops.to_frag16(rnd(N, K, seed=7, scale=0.1, dtype=torch.bfloat16)[pair_order(nH, nKV, d).to(DEV)].contiguous())
    for M in tokens:
        assert (M + 31) // 32 * ((N + 63) // 64) <= 256
        x = rnd(M, K, seed=M, dtype=torch.bfloat16)
        first = M // 3
        pos = torch.tensor([t if t < first else 5 + t - first for t in range(M)], dtype=torch.int32, device=DEV)
        seq = torch.tensor([1 if t < first else 0 for t in range(M)], dtype=torch.int32, device=DEV)
        n = int(pos.max()) + 1
        ang = torch.arange(n, dtype=torch.float64)[:, None] * 1e4 ** (-2.0 * torch.arange(d // 2, dtype=torch.float64) / d)
        cos, sin = torch.cos(ang).float().to(DEV), torch.sin(ang).float().to(DEV)
        got = []
        for fused in (False, True):
            kp, vp, bt = paged(n, nKV, d, torch.bfloat16, 2, seed=3)
            q = torch.full((M, nH * d), float("nan"), dtype=torch.bfloat16, device=DEV)
            if fused:
                ops.linear_rope_cache(acts_to_fragments(x), w, q, kp, vp, cos, sin, pos, seq, bt, k_in=K, num_heads=nH, num_kv_heads=nKV, head_dim=d,
                                      max_position=n - 1, kv_layout=layout, rows=M, x_layout=ops.LAYOUT_FRAG16)
            else:
                sums = torch.empty(M, N, dtype=torch.float32, device=DEV)
                ops.linear(acts_to_fragments(x), w, sums, n_out=N, k_in=K, layout=ops.LAYOUT_FRAG16, variant=ops.LINEAR_TILED_W16,
                           x_layout=ops.LAYOUT_FRAG16, rows=M, full_precision=False)
                ops.rope_cache_write(sums.to(torch.bfloat16), q, kp, vp, cos, sin, pos, seq, bt, num_heads=nH, num_kv_heads=nKV, head_dim=d,
                                     rotary_dim=d, max_position=n - 1, kv_layout=layout, interleaved=True)
            got.append((q, kp, vp))
        assert all(torch.equal(a, b) for a, b in zip(*got)), M
