"""32-bit products of up to sixteen tokens: at the edges of the rows a wave takes, the elements a step and the chunk that a block
keeps, in slices that end anywhere, against 64 bits and against the kernel for rows of any address; a token gets the same bits
whatever kernel its step's size brings about."""
import pytest
import torch
import torch.nn.functional as F

from alice_llm_amd.hip import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def rnd(*shape, seed=0, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(1, 1024), (17, 1028), (70, 2560), (46, 2564), (33, 5120), (18, 9220), (2304, 2048)])
@pytest.mark.parametrize("xdt,wdt", [("float32", "float32"), ("float32", "bfloat16"), ("bfloat16", "float32")])
def test_few_tokens(M, N, K, xdt, wdt):
    x, w = rnd(M, K, seed=M, dtype=DT[xdt]), rnd(N, K, seed=N, scale=0.1, dtype=DT[wdt])
    ref, tol = x.double() @ w.double().T, 8 * 0.1 * K * 2 ** -24           # (as in test_gpu_f32.py)
    moved = torch.empty(N * K + 1, dtype=w.dtype, device=DEV)[1:].view(N, K).copy_(w)
    for split in {1, 2, 3, 7, 8, ops.linear_split_hint(M, N, K, ops.LAYOUT_ROW)}:
        outs = []
        for wt in (w, moved):
            y = torch.full((split, M, N) if split > 1 else (M, N), float("nan"), device=DEV)
            ops.linear(x, wt, y, n_out=N, k_in=K, split_k=split, full_precision=True)
            outs.append(y.sum(0) if split > 1 else y)
            assert (outs[-1].double() - ref).abs().max() <= tol, split
    if N % 2 == 0:
        out = torch.full((M, N // 2), float("nan"), device=DEV)
        ops.linear(x, w, out, n_out=N // 2, k_in=K, epilogue=ops.EPI_GEGLU, full_precision=True)
        want = F.gelu(ref[:, :N // 2], approximate="tanh") * ref[:, N // 2:]
        assert ((out.double() - want).abs() <= 4 * tol + 1e-5 * want.abs()).all()
    capped = torch.full((M, N), float("nan"), device=DEV)
    ops.linear(x, w, capped, n_out=N, k_in=K, epilogue=ops.EPI_SOFTCAP, epi_param=5.0, full_precision=True)
    assert (capped.double() - 5 * torch.tanh(ref / 5)).abs().max() <= tol + 1e-5


@pytest.mark.parametrize("N,K,split", [(48, 1280, None), (700, 1408, None), (48, 1920, None), (64, 2304, None), (2304, 2048, 8), (40, 1030, 3), (40, 2000, 5)])
def test_slices_of_one_token(N, K, split):
    """A slice of one token's product is the product of that slice's elements, bit for bit: in the slices that the library plans
    (of which some end just below 512 elements) and in any others, at aligned and at odd addresses."""
    x, w = rnd(1, K, seed=1), rnd(N, K, seed=2, scale=0.1)
    moved = torch.empty(N * K + 1, device=DEV)[1:].view(N, K).copy_(w)
    split = split or ops.linear_split_hint(1, N, K, ops.LAYOUT_ROW)
    assert split > 1
    step = -(-(-(-K // split)) // 128) * 128
    for wt in (w, moved):
        y = torch.full((split, 1, N), float("nan"), device=DEV)
        ops.linear(x, wt, y, n_out=N, k_in=K, split_k=split, full_precision=True)
        for s in range(split):
            part, a, b = torch.zeros(1, N, device=DEV), s * step, min(K, (s + 1) * step)
            if a < b:
                ops.linear(x[:, a:b].contiguous(), w[:, a:b].contiguous(), part, n_out=N, k_in=b - a, full_precision=True)
            assert torch.equal(y[s], part), s


@pytest.mark.parametrize("M", [5, 8, 9, 12, 13, 16])
@pytest.mark.parametrize("N,K,splits", [(17, 1028, (1, 2)), (1002, 2048, (1, 4)),                     # four tokens a block
                                        (2050, 2564, (1,)), (4094, 1024, (1,)), (130, 9220, (1, 7)),   # quarters
                                        (4200, 1028, (1, 2)), (1100, 4100, (4, 8)),                   # eight rows a wave
                                        (2306, 3080, (5,)), (10310, 1284, (1,)), (25602, 1024, (1,))])       # eight waves a block
@pytest.mark.parametrize("xdt,wdt", [("float32", "float32"), ("float32", "bfloat16"), ("bfloat16", "float32")])
def test_five_to_sixteen_tokens(M, N, K, splits, xdt, wdt):
    x, w = rnd(M, K, seed=M, dtype=DT[xdt]), rnd(N, K, seed=N, scale=0.1, dtype=DT[wdt])
    ref, tol = x.double() @ w.double().T, 8 * 0.1 * K * 2 ** -24           # (as in test_gpu_f32.py)
    fours = [x[i:i + 4].contiguous() for i in range(0, M, 4)]

    def run(x, split=1, n=N, **epilogue):
        y = torch.full((split, x.shape[0], n) if split > 1 else (x.shape[0], n), float("nan"), device=DEV)
        ops.linear(x, w, y, n_out=n, k_in=K, split_k=split, full_precision=True, **epilogue)
        return y

    for split in splits:
        y = run(x, split)
        assert torch.equal(y, torch.cat([run(f, split) for f in fours], -2)), split
        assert ((y.sum(0) if split > 1 else y).double() - ref).abs().max() <= tol, split
    for e, n in ((dict(epilogue=ops.EPI_GEGLU), N // 2), (dict(epilogue=ops.EPI_SOFTCAP, epi_param=5.0), N)):
        if N % 2 == 0 or n == N:
            assert torch.equal(run(x, n=n, **e), torch.cat([run(f, n=n, **e) for f in fours]))


def test_a_token_gets_the_same_with_and_without_others():
    """One token (a wave a row, or four rows a wave in large matrices) and up to sixteen: the same bits, whole and in the slices that
    the library plans for two to sixteen tokens (one number; for one token it may be another)."""
    for N, K in ((40, 1028), (2304, 2304), (8200, 2560), (4096, 2304)):
        x, w = rnd(16, K, seed=1), rnd(N, K, seed=2)
        hints = {ops.linear_split_hint(M, N, K, ops.LAYOUT_ROW) for M in range(2, 17)}
        assert len(hints) == 1
        for split in {1} | hints:
            short = split > 1 and -(-K // split) <= 384
            outs = []
            for M in (16, 1, 2, 4, 5, 7, 8, 9, 12, 13):
                y = torch.empty((split, M, N) if split > 1 else (M, N), device=DEV)
                ops.linear(x[:M].contiguous(), w, y, n_out=N, k_in=K, split_k=split, full_precision=True)
                outs.append(y)
            # (slices of up to 384 elements: two and more tokens as columns of the matrix instruction, one as ever)
            for y in outs[1:]:
                M = y.shape[-2]
                assert (M == 1 and short) or torch.equal(y, outs[0][..., :M, :]), (N, K, split, M)


@pytest.mark.parametrize("M,N", [(3, 12), (16, 12), (8, 2060), (16, 2060), (8, 4300), (12, 4300), (16, 4300), (16, 10400)])
def test_weights_that_are_no_numbers_stay_in_their_rows(M, N):
    """What is read again behind a row's end is not multiplied: a last element that is infinite reaches its own product alone."""
    x, w = rnd(M, 2308, seed=1), rnd(N, 2308, seed=2)
    x[:, -1] = 0.0
    x[1, -1] = 1.0
    w[5, -1] = float("inf")
    x[2, -1] = float("inf")
    y = torch.empty(M, N, device=DEV)
    ops.linear(x, w, y, n_out=N, k_in=2308, full_precision=True)
    want = x.double() @ w.double().T
    assert torch.equal(torch.isnan(y).cpu(), torch.isnan(want).cpu()) and torch.equal(torch.isinf(y).cpu(), torch.isinf(want).cpu())


def test_short_prompts_captured_and_eagerly():
    """Prompts of two to sixteen tokens, which a captured step rounds to sixteen: the same bits."""
    import alice_llm_amd as alice
    from helpers import TINY, random_tokens
    raw = dict(TINY["tiny-a"][0], num_hidden_layers=1, hidden_size=1024, intermediate_size=1024)
    model = alice.Model.random(raw, seed=4, dtype="float32", fast=True)
    eager, graph = (model.engine(max_tokens=64 * 8, max_seqs=2, use_graphs=g) for g in (False, True))
    assert graph.capture_prompts
    for n in (2, 3, 4, 5, 9, 15, 16):
        replayed = []
        toks = random_tokens(256, n, n)
        for _ in range(4):                                               # seen, captured, replayed
            a, b = eager.open(1), graph.open(1)
            want = eager.step(a, [toks], "last")
            replayed.append(graph.step(b, [toks], "last"))
            assert torch.equal(replayed[-1], want), n
            eager.close(a), graph.close(b)
