"""Float32 products on the bfloat16 matrix instruction (operands in three parts): every tile at its edges, against 64 bits; precision
against the 32-bit instruction; numbers that have no three parts."""
import pytest
import torch
import torch.nn.functional as F

from alice_llm_amd.hip import ops
from test_gpu_kernels import rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"


def product(x, w, split=1, epi=ops.EPI_NONE, param=0.0):
    M, K = x.shape
    N = w.shape[0] // (2 if epi == ops.EPI_GEGLU else 1)
    y = torch.full(((split,) if split > 1 else ()) + (M, N), float("nan"), device=DEV)
    ops.linear(x, w, y, n_out=N, k_in=K, epilogue=epi, epi_param=param, split_k=split, full_precision=True)
    return y


def bound(x, w):
    """What any order of the six products' sums may be off: 2^-23 of every product left out, and six roundings for 32 elements and
    one for each part's sum, of at most 2^-23 (the instruction adds without rounding to nearest) of all products' sizes."""
    K = x.shape[1]
    return (x.double().abs() @ w.double().abs().T) * 2.0 ** -23 * (1 + 6 * (K // 32 + 2) + 8)


# tokens, rows, inner elements, slices: tiles 0 .. 5; last rows and tokens of a tile missing, an inner dimension that is no multiple
# of 32 or of 64, groups of unequally many stages, rows that are no multiple of 16 bytes of outputs
CASES = [(128, 16384, 2304, 1), (500, 9217, 2304, 1), (500, 4096, 2304, 1), (497, 4095, 2308, 1), (500, 2304, 9216, 3), (500, 2302, 9220, 6),
         (33, 2304, 9216, 4), (19, 2303, 9212, 8), (17, 2304, 2048, 7), (65, 1000, 16384, 8), (300, 20000, 164, 1), (2000, 1152, 1156, 2)]


@pytest.mark.parametrize("M,N,K,split", CASES)
def test_products_in_thirds(M, N, K, split):
    assert ops.linear_thirds_tile(M, N, K, False, split) >= 0
    x, w = rnd(M, K, seed=M), rnd(N, K, seed=N, scale=0.1)
    got, ref = product(x, w, split), x.double() @ w.double().T
    got = got.double().sum(0) if split > 1 else got.double()
    assert torch.isfinite(got).all() and ((got - ref).abs() <= bound(x, w)).all()
    if split == 1:
        cap = product(x, w, 1, ops.EPI_SOFTCAP, 2.0)
        assert ((cap.double() - 2 * torch.tanh(ref / 2)).abs() <= bound(x, w) + 1e-6).all()


def test_every_tile_is_among_the_cases():
    assert {ops.linear_thirds_tile(M, N, K, False, s) for M, N, K, s in CASES} == {0, 1, 2, 3, 4, 5}


GATED = [(500, 9216, 2304), (497, 9212, 2308), (500, 4610, 2304), (128, 9218, 2304), (64, 9218, 2304), (2048, 1025, 2304),
         (300, 5000, 2308), (65, 2305, 2308), (19, 14336, 2304)]


@pytest.mark.parametrize("M,N,K", GATED)
def test_gated_products_in_thirds(M, N, K):
    assert ops.linear_thirds_tile(M, N, K, True) >= 0
    x, w = rnd(M, K, seed=M), rnd(2 * N, K, seed=N, scale=0.02)
    got, off = product(x, w, epi=ops.EPI_GEGLU).double(), bound(x, w)
    ref = x.double() @ w.double().T
    g, u = ref[:, :N], ref[:, N:]
    # the gate's slope is at most 1.13; 1e-6 for the 32-bit function itself
    assert ((got - F.gelu(g, approximate="tanh") * u).abs() <= 1.13 * off[:, :N] * u.abs() + off[:, N:] * g.abs() + 1e-6 * (1 + g.abs() * u.abs())).all()


def single(M, K, seed):
    """Tokens of one element each, the others zeros, in places all over the inner dimension."""
    gen = torch.Generator().manual_seed(seed)
    x = torch.zeros(M, K)
    x[torch.arange(M), (torch.arange(M) * K // M + torch.randint(0, max(1, K // M), (M,), generator=gen)).clamp(max=K - 1)] = torch.randn(M, generator=gen)
    x[0] = x[M - 1] = 0.0
    x[0, 0], x[M - 1, K - 1] = 1.7, -1.3
    return x.to(DEV)


# One product alone: three parts' products left out, 2^-24 of it at most, and the sum of the largest one and the others rounded to nearest,
# 2^-24; the others are 2^-6.5 of it at most and are cut off five times, at 2^-23 of themselves.  Without x0 w2 or x2 w0 it would be off by
# up to 2^-17, without x1 w1 by up to 2^-16.
ALONE = 2.0 ** -23 * 1.06


@pytest.mark.parametrize("M,N,K,split", CASES)
def test_single_products(M, N, K, split):
    """All six products are there, at every tile and wherever in the inner dimension."""
    assert ops.linear_thirds_tile(M, N, K, False, split) >= 0
    x, w = single(M, K, M), rnd(N, K, seed=N)
    got, ref = product(x, w, split), x.double() @ w.double().T
    got = got.double().sum(0) if split > 1 else got.double()
    assert ((got - ref).abs() <= ALONE * ref.abs()).all()


@pytest.mark.parametrize("M,N,K", GATED)
def test_single_gated_products(M, N, K):
    assert ops.linear_thirds_tile(M, N, K, True) >= 0
    x, w = single(M, K, M), rnd(2 * N, K, seed=N)
    got, ref = product(x, w, epi=ops.EPI_GEGLU).double(), x.double() @ w.double().T
    g, u = ref[:, :N], ref[:, N:]
    assert ((got - F.gelu(g, approximate="tanh") * u).abs() <= 2.13 * ALONE * (g * u).abs() + 1e-6 * (1 + (g * u).abs())).all()


def on_the_32_bit_instruction(x, w, split=1, epi=ops.EPI_NONE):
    """The same product over rows of one more element that is zero: rows that are no multiple of four elements take that instruction."""
    return product(*(F.pad(a, (0, 1)).contiguous() for a in (x, w)), split, epi)


@pytest.mark.parametrize("M,N,K,split", CASES)
@pytest.mark.parametrize("spread", [0.0, 3.0])
def test_every_tile_is_no_less_precise_than_the_32_bit_instruction(M, N, K, split, spread):
    x, w = (rnd(n, K, seed=i) * torch.exp(spread * rnd(n, K, seed=i + 2)) for i, n in enumerate((M, N)))
    ref = x.double() @ w.double().T
    err = [float((y.double().sum(0) if split > 1 else y.double()).sub(ref).norm() / ref.norm())
           for y in (product(x, w, split), on_the_32_bit_instruction(x, w, split))]
    assert err[0] <= err[1], err


@pytest.mark.parametrize("M,N,K,split", [(500, 4096, 2304, 1), (500, 9217, 2304, 1), (500, 2304, 9216, 3), (65, 1000, 16384, 8)])
@pytest.mark.parametrize("elements", [1, 2, 4, 16, 64, 256])
def test_tokens_of_few_elements(M, N, K, split, elements):
    """Sums of few products, which leave nothing to average, against the 32-bit instruction, which rounds once a product.  A product of two
    normal numbers is rounded by 2.5e-8 of it in the mean, the products left out are 2^-25 sqrt(2) / 3 of it for mantissas of 1, 0.6e-8
    in the mean: 3 % more where the sums themselves round next to nothing (a slice has one to three of them), less from then on."""
    assert ops.linear_thirds_tile(M, N, K, False, split) >= 0
    gen = torch.Generator().manual_seed(elements)
    at = torch.rand(M, K, generator=gen).argsort(1)[:, :elements]
    x, w = torch.zeros(M, K).scatter_(1, at, torch.randn(M, elements, generator=gen)).to(DEV), rnd(N, K, seed=N)
    ref = x.double() @ w.double().T
    err = [float((y.double().sum(0) if split > 1 else y.double()).sub(ref).norm() / ref.norm())
           for y in (product(x, w, split), on_the_32_bit_instruction(x, w, split))]
    assert err[0] <= (1.05 if elements <= 3 * split else 1.0) * err[1], err


@pytest.mark.parametrize("M,N,K", GATED)
def test_gated_products_are_no_less_precise_than_the_32_bit_instruction(M, N, K):
    x, w = rnd(M, K, seed=M), rnd(2 * N, K, seed=N, scale=0.1)
    g, u = (x.double() @ w.double().T).chunk(2, 1)
    ref = F.gelu(g, approximate="tanh") * u
    err = [float((y.double() - ref).norm() / ref.norm()) for y in (product(x, w, epi=ops.EPI_GEGLU), on_the_32_bit_instruction(x, w, epi=ops.EPI_GEGLU))]
    assert err[0] <= err[1], err


@pytest.mark.parametrize("M,N,K,split", [(500, 4096, 2304, 1), (500, 2304, 9216, 3), (500, 20000, 164, 1), (128, 2304, 16384, 8)])
@pytest.mark.parametrize("spread", [0.0, 3.0])
def test_no_less_precise_than_the_32_bit_instruction(M, N, K, split, spread):
    """Normal numbers, and numbers whose sizes are spread over some orders of magnitude.  The same product over rows of one more element
    that is zero takes the 32-bit instruction (rows that are no multiple of four elements)."""
    assert ops.linear_thirds_tile(M, N, K, False, split) >= 0
    x, w = (rnd(n, K, seed=i) * torch.exp(spread * rnd(n, K, seed=i + 2)) for i, n in enumerate((M, N)))
    ref = x.double() @ w.double().T
    err = [float((y.double().sum(0) if split > 1 else y.double()).sub(ref).norm() / ref.norm())
           for y in (product(x, w, split), product(*(F.pad(a, (0, 1)).contiguous() for a in (x, w)), split))]
    assert err[0] <= err[1], err
    # and not in one direction: the mean over the tokens is no larger than that of errors of either sign (five standard deviations)
    e = (product(x, w, split).double().sum(0) if split > 1 else product(x, w, split).double()) - ref
    assert float(e.mean(0).norm()) <= 1.5 * float(e.norm()) / M, (float(e.mean(0).norm()), float(e.norm()) / M)


def test_what_has_no_three_parts():
    """Infinities, no numbers, numbers that round to no finite bfloat16, and sums of numbers so small that their last part is below
    the smallest bfloat16: what 32-bit products give."""
    M, N, K = 500, 4096, 2304
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=0.02)
    x[3, 7], x[200, 2300], x[201, 5] = float("inf"), float("-inf"), float("nan")
    w[17, 9], w[4000, 0] = float("inf"), float("nan")
    x[77] = 0.0
    x[90, 100] = 3.4e38
    w[:, 100] *= 1e-3
    got, ref = product(x, w), x.double() @ w.double().T
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    ok = torch.isfinite(ref)
    assert torch.equal(got[~ok & ~torch.isnan(ref)].double(), ref[~ok & ~torch.isnan(ref)])
    x2, w2 = (torch.where(torch.isfinite(a), a, 0.0) for a in (x, w))
    assert ((got.double() - ref).abs()[ok] <= (bound(x2, w2) * 16)[ok]).all()      # (32 roundings for 32 elements instead of 6)
    tiny = rnd(M, K, seed=3) * 1e-34
    got, ref = product(tiny, w[:, :].nan_to_num(0.0, 0.0, 0.0)), tiny.double() @ w.nan_to_num(0.0, 0.0, 0.0).double().T
    assert ((got.double() - ref).norm() <= 1e-5 * ref.norm())
    assert (product(torch.zeros(M, K, device=DEV), w2) == 0).all()


@pytest.mark.parametrize("ex,ew", [(-112, 60), (60, -112), (-120, 21), (-110, 100)])
def test_small_numbers_times_large_ones(ex, ew):
    """The last parts of the small factor are below the smallest normal bfloat16 while the sums are ordinary numbers."""
    M, N, K = 500, 4096, 2304
    x, w = torch.ldexp(rnd(M, K, seed=4), torch.tensor(ex, device=DEV)), torch.ldexp(rnd(N, K, seed=5), torch.tensor(ew, device=DEV))
    got, ref = product(x, w).double(), x.double() @ w.double().T
    assert ((got - ref).abs() <= 16 * bound(x, w)).all()          # (32 roundings for 32 elements instead of 6)
    assert float((got - ref).norm() / ref.norm()) <= 1e-5


def test_a_token_depends_on_no_other_and_captured_steps_add_as_eager_ones():
    M, N, K = 129, 9216, 2304
    x, w = rnd(192, K, seed=1), rnd(N, K, seed=2)
    all_rows = product(x, w)
    for n in (M, 144, 191):                                       # one multiple of 64: one tile, one order
        assert torch.equal(product(x[:n].contiguous(), w), all_rows[:n])
    y = torch.empty(192, N, device=DEV)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        ops.linear(x, w, y, n_out=N, k_in=K, full_precision=True)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            ops.linear(x, w, y, n_out=N, k_in=K, full_precision=True)
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, all_rows)


@pytest.mark.parametrize("M,N,K,split", [c for c in CASES if c[0] >= 17])
@pytest.mark.parametrize("odd", [float("nan"), float("-inf"), 2.0 ** 21, 2.0 ** -80])
def test_tokens_beside_one_that_has_no_three_parts(M, N, K, split, odd):
    """A token with a number that sends its sums to the 32-bit instruction (a token of tiny numbers: tiny sums) changes no other token's
    bits, a row of W with one no other output's."""
    x, w = rnd(M, K, seed=M), rnd(N, K, seed=N, scale=0.1)
    plain = product(x, w, split)
    x2, w2, token, row = x.clone(), w.clone(), M // 2, N // 3
    if odd < 1 and odd > 0:
        x2[token] *= odd
        w2[row] *= odd
    else:
        x2[token, K // 3] = w2[row, K - 1] = odd
    got = product(x2, w, split)
    keep = [t for t in range(M) if t != token]
    assert torch.equal(got[..., keep, :], plain[..., keep, :]) and not torch.equal(got[..., token, :], plain[..., token, :])
    # and what the token gets does not hang on who its neighbours are
    assert torch.equal(product(x2.flip(0).contiguous(), w, split)[..., M - 1 - token, :].nan_to_num(7.0), got[..., token, :].nan_to_num(7.0))
    got = product(x, w2, split)
    keep = [n for n in range(N) if n != row]
    assert torch.equal(got[..., keep], plain[..., keep]) and not torch.equal(got[..., row], plain[..., row])


@pytest.mark.parametrize("M,N,K,split", [(500, 4096, 2304, 1), (500, 2304, 9216, 3), (17, 2304, 2048, 7), (128, 16384, 2304, 1)])
def test_sums_of_zero(M, N, K, split):
    """Factors of which no part is left give zeros that are none; tokens and rows of zeros, and pairs that cancel, give zeros."""
    assert ops.linear_thirds_tile(M, N, K, False, split) >= 0
    x, w = rnd(M, K, seed=M, scale=2.0 ** 17).clamp(-2.0 ** 20, 2.0 ** 20), rnd(N, K, seed=N)
    few = torch.zeros_like(x)
    few[3, :] = torch.ldexp(rnd(K, seed=3), torch.tensor(-138, device=DEV))      # subnormal, less than any bfloat16
    few[5, ::16] = x[5, ::16]
    few[9, 1] = x[9, 1]
    few[11, 0], few[11, 1] = 3.0 * 2.0 ** -116 * (1 + 2.0 ** -22), -3.0 * 2.0 ** -116      # what is left of the sum is a lost part
    w[:, 1] = w[:, 0]
    w[4], w[7] = 0.0, torch.ldexp(rnd(K, seed=7), torch.tensor(-139, device=DEV))
    big = w * 2.0 ** 17
    for a, b in ((few, big.clamp(-2.0 ** 20, 2.0 ** 20)), (x, w)):
        got, ref = product(a, b, split), a.double() @ b.double().T
        got = got.double().sum(0) if split > 1 else got.double()
        assert ((got - ref).abs() <= 16 * bound(a, b) + 2.0 ** -140).all()
        assert torch.equal(got == 0, ref.abs() < 2.0 ** -150)      # (a token and a row of such numbers: less than any float32)
    # the token of what is left is the only difference
    other = few.clone()
    other[3] = other[11] = 0.0
    b = big.clamp(-2.0 ** 20, 2.0 ** 20)
    keep = [t for t in range(M) if t not in (3, 11)]
    assert torch.equal(product(other, b, split)[..., keep, :], product(few, b, split)[..., keep, :])
