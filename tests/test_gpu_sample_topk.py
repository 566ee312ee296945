"""Top-k of up to 200 in one pass over the row: against the plain sampler, at the edges of chunks, tiles and lists."""
import math

import pytest
import torch

from alice_llm_amd.hip import ops
from test_gpu_kernels import DEV, check_samples, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,V", [(1, 300), (3, 4095), (3, 4096), (2, 16388), (65, 16385), (1, 256000), (3, 524288), (2, 524292)])
@pytest.mark.parametrize("top_k,top_p", [(1, 1.0), (37, 0.7), (200, 0.95), (201, 0.95)])
def test_small_k_at_the_edges(B, V, top_k, top_p):
    g = torch.Generator().manual_seed(V + top_k)
    spread = rnd(B, V, seed=V, scale=3.0)
    for logits in (spread, spread.sort(dim=1).values, spread.sort(dim=1, descending=True).values):
        check_samples(logits, torch.rand(B, generator=g), 0.8, top_k, top_p)


def test_lists_that_outgrow_their_room_and_rows_without_a_finite_maximum():
    """All large values in one thread's places, thousands of ties, masked rows and rows with an infinite logit beside an
    ordinary row: each row gets what it gets alone."""
    V, g = 70000, torch.Generator().manual_seed(5)
    ordinary = rnd(1, V, seed=31, scale=2.0)
    uneven = rnd(1, V, seed=32, scale=0.1)
    uneven[0, torch.arange(0, 16384, 1024)] += 9.0                    # 16 of thread 0's 64 elements of the first chunk
    uneven[0, 1:4] += 9.0
    ties = (rnd(1, V, seed=33) > 0.5).float()
    masked = torch.full((1, V), -math.inf, device=DEV)
    masked[0, [5, 69999]] = torch.tensor([1.0, 0.5], device=DEV)
    top = rnd(1, V, seed=34)
    top[0, 777] = 1e30
    rows = torch.cat([ordinary, uneven, ties, masked, top])
    for top_k, top_p in ((20, 0.9), (3, 1.0), (150, 0.5)):
        u = torch.rand(5, generator=g)
        got = check_samples(rows, u, 1.0, top_k, top_p)
        assert got == [ops.sample(rows[i:i + 1], u[i:i + 1].to(DEV), 1.0, top_k, top_p).item() for i in range(5)]
        assert got[3] in (5, 69999) and got[4] == 777
