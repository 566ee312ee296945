"""Products in tiles of 256 tokens: edges of tiles, k-tiles a slice, what the launcher takes them for and what it refuses."""
import math

import pytest
import torch

from alice_llm_amd.hip import ops
from test_gpu_kernels import acts_from_fragments, acts_to_fragments, close, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"
TILES = {256: ops.LINEAR_LARGE_256, 192: ops.LINEAR_LARGE_192, 128: ops.LINEAR_LARGE_128}


def product(x, wf, M, N, K, split=1, **kw):
    y = torch.full((split, M, N) if split > 1 else (M, N), float("nan"), dtype=torch.float32, device=DEV)
    ops.linear(acts_to_fragments(x), wf, y, n_out=N, k_in=K, layout=ops.LAYOUT_FRAG16, split_k=split, full_precision=False, rows=M,
               x_layout=ops.LAYOUT_FRAG16, **kw)
    return y


# tokens around a tile's and a 16-token tile's edge, features beyond one tile, inner dimensions of two pairs of k-tiles and more, more tiles than
# blocks (the last two sizes: 270 and more), slices of unlike lengths (1,280: 14, 14 and 12 k-tiles)
@pytest.mark.parametrize("features", [256, 192, 128])
@pytest.mark.parametrize("M,N,K,split", [(1, 16, 128, 1), (15, 400, 192, 1), (256, 256, 128, 1), (257, 528, 384, 2), (300, 2304, 512, 4), (513, 272, 1280, 3),
                                         (1100, 7440, 128, 1), (2049, 4112, 256, 2)])
def test_sums_are_those_of_the_tiled_kernel(features, M, N, K, split):
    """The same bits: a slice's k-tiles are added in their order by either kernel."""
    x, wf = rnd(M, K, seed=1, dtype=torch.bfloat16), rnd(N, K, seed=2, scale=0.1, dtype=torch.bfloat16)
    ref = x.double() @ wf.double().T
    wf = ops.to_frag16(wf)
    y = product(x, wf, M, N, K, split, variant=TILES[features])
    assert torch.equal(y, product(x, wf, M, N, K, split, variant=ops.LINEAR_MFMA))
    close(y.sum(0) if split > 1 else y, ref, 2e-4 * math.sqrt(K / 64), 1e-5)


@pytest.mark.parametrize("features", [256, 192, 128])
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (130, 208, 192), (257, 1040, 256), (700, 9280, 128)])
@pytest.mark.parametrize("form", [0.0, ops.GATED_SILU])
def test_gated_products(features, M, N, K, form):
    x, w = rnd(M, K, seed=3, dtype=torch.bfloat16), rnd(2 * N, K, seed=4, scale=0.3, dtype=torch.bfloat16)
    g, u = x.double() @ w.double()[:N].T, x.double() @ w.double()[N:].T
    ref = (torch.nn.functional.gelu(g, approximate="tanh") if form == 0.0 else torch.nn.functional.silu(g)) * u
    wf, outs = ops.to_frag16(w), []
    for variant in (TILES[features], ops.LINEAR_MFMA):
        for frag in ((True, False) if N % 32 == 0 else (False,)):
            size = -(-M // 16) * 16 * N if frag else (M, N)
            y = torch.full((size,) if frag else size, float("nan"), dtype=torch.bfloat16, device=DEV)
            ops.linear(acts_to_fragments(x), wf, y, n_out=N, k_in=K, layout=ops.LAYOUT_FRAG16, epilogue=ops.EPI_GEGLU, epi_param=form,
                       variant=variant, full_precision=False, rows=M, x_layout=ops.LAYOUT_FRAG16,
                       y_layout=ops.LAYOUT_FRAG16 if frag else ops.LAYOUT_ROW)
            outs.append(acts_from_fragments(y, M, N).to(DEV) if frag else y)
    assert all(torch.equal(o, outs[0]) for o in outs)
    close(outs[0], ref, 2e-2 * math.sqrt(K / 64), 2 ** -7)


def test_infinities_stay_in_their_token_and_feature():
    M, N, K = 260, 272, 256
    x, w = rnd(M, K, seed=5, dtype=torch.bfloat16), rnd(N, K, seed=6, dtype=torch.bfloat16)
    x[259, 7], w[270, 200] = float("inf"), float("nan")
    y = product(x, ops.to_frag16(w), M, N, K, variant=ops.LINEAR_LARGE_256)
    odd = torch.zeros(M, N, dtype=torch.bool, device=DEV)
    odd[259], odd[:, 270] = True, True
    assert torch.equal(~torch.isfinite(y), odd)


def test_what_it_does_not_take():
    x = rnd(20, 160, seed=7, dtype=torch.bfloat16)
    for N, K, split in ((32, 160, 1), (40, 128, 1), (32, 128, 2), (32, 64, 1)):      # an odd number of k-tiles, a part of a tile, single pairs
        w = ops.to_frag16(rnd(N, K, seed=8, dtype=torch.bfloat16))
        with pytest.raises(ops.HipLibraryError, match="tiles of 256 tokens"):
            product(x[:, :K].contiguous(), w, 20, N, K, split, variant=ops.LINEAR_LARGE_128)
    w = ops.to_frag16(rnd(32, 128, seed=8, dtype=torch.bfloat16))
    y = torch.empty(20, 32, dtype=torch.float32, device=DEV)
    with pytest.raises(ops.HipLibraryError, match="tiles of 256 tokens"):            # activations in rows
        ops.linear(x[:, :128].contiguous(), w, y, n_out=32, k_in=128, layout=ops.LAYOUT_FRAG16, variant=ops.LINEAR_LARGE_256, full_precision=False)


@pytest.mark.parametrize("M", [447, 448, 1000, 2048])
@pytest.mark.parametrize("N,K", [(2304, 9216), (2304, 2048), (4096, 2304)])
def test_the_proposed_slices_have_the_tiled_kernels_bits(M, N, K):
    """(Which kernel takes them does not show in the bits: test_product_slices.py asks the rule.)"""
    x, w = rnd(M, K, seed=9, dtype=torch.bfloat16), rnd(N, K, seed=10, dtype=torch.bfloat16)
    split = ops.linear_split_hint(M, N, K, ops.LAYOUT_FRAG16)
    wf = ops.to_frag16(w)
    y = product(x, wf, M, N, K, split)
    assert torch.equal(y, product(x, wf, M, N, K, split, variant=ops.LINEAR_MFMA))
