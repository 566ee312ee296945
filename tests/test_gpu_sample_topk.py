"""Top-k of up to 200 in one pass over the row: against the plain sampler, at the edges of chunks, tiles and lists."""
import math
import random

import pytest
import torch

from alice_llm_amd.hip import ops
from alice_llm_amd.sampling.sampler import Sampler, uniforms
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
    """All large values in one thread's places, thousands of ties, a masked row, one with a huge logit, with an infinite one and with
    one that is no number, beside an ordinary row: each row gets what it gets alone."""
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
    odd = rnd(2, V, seed=35)
    odd[0, 30000], odd[1, 40000] = math.inf, math.nan
    rows = torch.cat([ordinary, uneven, ties, masked, top])
    for top_k, top_p in ((20, 0.9), (3, 1.0), (150, 0.5)):
        u = torch.rand(7, generator=g)
        got = check_samples(rows, u[:5], 1.0, top_k, top_p)
        both = torch.cat([odd[:1], rows, odd[1:]])
        order = [5, 0, 1, 2, 3, 4, 6]
        many = ops.sample(both, u[order].to(DEV), 1.0, top_k, top_p).tolist()
        assert many[1:6] == got and all(0 <= t < V for t in many)
        assert many == [ops.sample(both[i:i + 1], u[order[i]:order[i] + 1].to(DEV), 1.0, top_k, top_p).item() for i in range(7)]
        assert got[3] in (5, 69999) and got[4] == 777


@pytest.mark.parametrize("mask", [-math.inf, -1e9, torch.finfo(torch.float32).min])
@pytest.mark.parametrize("B,V", [(2, 70000), (1, 256000), (70, 66001)])
def test_masked_rows_are_settled_without_their_masked_elements(mask, B, V):
    """Chunks that hold nothing but masked elements, or few others: spread, side by side, in one thread's places, fewer than k of
    them, in the last chunk alone, and as many as fill a list.  The draw is the plain one, and takes no longer than a row without a
    mask does by more than the second look at the chunks (a row bisected whole takes fifty times as long)."""
    g = torch.Generator().manual_seed(V)
    spread = torch.randperm(V, generator=g)
    base = rnd(B, V, seed=3, scale=3.0)
    sets = [spread[:1000], torch.arange(5000, 6000), torch.arange(0, V, 1024), spread[:4], torch.arange(V - 90, V), torch.arange(V // 2),
            spread[:V // 3], torch.arange(4)]

    def time(rows, u, k):
        ops.sample(rows, u, 0.8, k, 0.95)
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(5):
            ops.sample(rows, u, 0.8, k, 0.95)
        b.record()
        b.synchronize()
        return a.elapsed_time(b)

    for keep in sets:
        rows = torch.full_like(base, mask)
        rows[:, keep.to(DEV)] = base[:, keep.to(DEV)]
        for top_k in (5, 50, 150):
            u = torch.rand(B, generator=g)
            got = ops.sample(rows, u.to(DEV), 0.8, top_k, 0.95).tolist()
            assert set(got) <= set(keep.tolist()) and got[:4] == check_samples(rows[:4], u[:4], 0.8, top_k, 0.95)
            assert min(time(rows, u.to(DEV), top_k) for _ in range(3)) < 8 * time(base, u.to(DEV), top_k), (len(keep), top_k)


@pytest.mark.parametrize("ties", [100, 128, 129, 257, 513, 1000, 1030])
@pytest.mark.parametrize("V", [40000, 300001])
def test_as_many_tied_at_the_threshold_as_change_the_shares_of_a_survivor(ties, V):
    """The rows' block gives a survivor 8, 4, 2 or 1 of its threads; ties at the threshold are all kept, many of them in one lane's
    share of a tile."""
    g = torch.Generator().manual_seed(ties)
    logits = rnd(4, V, seed=ties, scale=0.5).clamp_(max=1.9)
    logits[0, torch.randperm(V, generator=g)[:ties].to(DEV)] = 3.0
    logits[1, 4000:4000 + ties] = 3.0
    logits[2, torch.arange(ties, device=DEV) * 8] = 3.0
    logits[3, V - ties:] = 3.0
    logits[:, 17] = 4.0
    for top_k, top_p in ((2, 1.0), (20, 0.6)):
        check_samples(logits, torch.rand(4, generator=g), 0.7, top_k, top_p)


@pytest.mark.parametrize("n", [1, 30, 256, 257])
@pytest.mark.parametrize("seed", [0, -3, 2 ** 70 + 5])
def test_uniform_numbers_made_by_the_launch_are_those_of_the_sampler(n, seed):
    """Rows whose numbers the launch makes itself, and those that go the other way (many rows, numbers of another type or below 0),
    draw as they do with the sampler's own numbers."""
    rng = random.Random(n)
    logits = rnd(n, 5000, seed=n)
    draws = [rng.randrange(10000) for _ in range(n)]
    for requests in ([rng.randrange(2 ** 64) for _ in range(n)], [-1] * n, [2 ** 64 + 3] * n, [True] * n):
        u = uniforms(seed, requests, draws).to(DEV)
        for top_k, top_p in ((0, 1.0), (50, 0.9), (0, 0.9)):
            assert Sampler(0.9, top_k, top_p, seed=seed)(logits, requests, draws).tolist() == ops.sample(logits, u, 0.9, top_k, top_p).tolist()
    if n > 1:
        with pytest.raises(ops.HipLibraryError):
            Sampler(0.9, seed=seed)(logits, [1] * (n - 1), [1] * (n - 1))
    with pytest.raises(TypeError):
        Sampler(0.9, seed=seed)(logits, [1.5] * n, draws)


@pytest.mark.parametrize("V", [24000, 36864, 40000, 49152, 61000, 151936])
def test_rows_of_any_number_of_chunks_are_settled(V):
    """6, 9, 10, 12 and 15 chunks, and 10 of four tiles: the rows' block finds a bound that at most 1,024 elements reach whatever its
    waves' shares of the chunks are.  Then it takes the time that it takes for 16 chunks with the same k, which are the same phases over as
    many elements (14 us with a k of 20, 34 with 200; the chunks' own kernel adds at most 3 us for four tiles a chunk).  A row that is
    bisected whole takes 90 us more."""
    u = torch.rand(2, generator=torch.Generator().manual_seed(V))
    logits, even = rnd(2, V, seed=V, scale=4.0), rnd(2, 65536, seed=V, scale=4.0)

    def time(rows, k):
        dev = u.to(DEV)
        ops.sample(rows, dev, 0.8, k, 0.95)
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(20):
            ops.sample(rows, dev, 0.8, k, 0.95)
        b.record()
        b.synchronize()
        return a.elapsed_time(b) / 20

    for top_k in (145, 175, 200):
        check_samples(logits, u, 0.8, top_k, 0.95)
        same, this = min(time(even, top_k) for _ in range(3)), min(time(logits, top_k) for _ in range(3))
        assert this < same + 0.04, (top_k, same, this)
