"""The streaming product's slices of the inner dimension where rounding up leaves the last ones without elements: every slice's own sum."""
import pytest
import torch

from alice_llm_amd.hip import ops
from alice_llm_amd.parts.base import Precision
from alice_llm_amd.parts.linear import Linear
from test_gpu_kernels import acts_to_fragments, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"


def slices_of(K, split):
    per = -(-(-(-K // 32)) // split) * 32
    return [(min(K, z * per), min(K, (z + 1) * per)) for z in range(split)]


def check(y, x, w, K, split):
    for z, (a, b) in enumerate(slices_of(K, split)):
        xs, ws = x[:, a:b].double(), w[:, a:b].double()
        # products of bfloat16 numbers are exact in 32 bits: as many additions as elements, of at most 2^-23 of all products' sizes
        assert ((y[z].double() - xs @ ws.T).abs() <= (b - a) * 2.0 ** -23 * (xs.abs() @ ws.abs().T)).all(), z


# The last slice with elements: a whole one before empty ones (k-tiles 25 / 35 / 135 / 1089), a rest before empty ones (33 / 132 / 31),
# a rest that is the last slice (29), a whole last slice (64).  More than one k-tile a wave everywhere, eight waves a block at 1089.
@pytest.mark.parametrize("K,split,empty", [(800, 6, 1), (1120, 8, 1), (4320, 16, 1), (1056, 8, 1), (4224, 16, 1), (992, 7, 0), (928, 5, 0), (2048, 4, 0),
                                           (34848, 34, 1)])
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
def test_whole_partial_and_empty_last_slices(K, split, empty, M):
    assert (sum(a == b for a, b in slices_of(K, split)) > 0) == bool(empty)
    N = 1024 if K < 30000 else 144
    x, w = rnd(M, K, seed=M, dtype=torch.bfloat16), rnd(N, K, seed=K, scale=0.1, dtype=torch.bfloat16)
    wf = ops.to_frag16(w)
    for layout, acts in ((ops.LAYOUT_ROW, x), (ops.LAYOUT_FRAG16, acts_to_fragments(x))):
        y = torch.full((split, M, N), float("nan"), dtype=torch.float32, device=DEV)
        ops.linear(acts, wf, y, n_out=N, k_in=K, layout=ops.LAYOUT_FRAG16, split_k=split, variant=ops.LINEAR_SKINNY, full_precision=False, rows=M,
                   x_layout=layout)
        check(y, x, w, K, split)


@pytest.mark.parametrize("M,N,K", [(17, 1024, 4224), (64, 1024, 4304), (8, 1024, 5760), (40, 1280, 3080), (33, 1280, 3072)])
def test_the_slices_that_a_projection_of_rows_takes(M, N, K):
    """A projection asks for as many slices as activations in fragment order would have; rows go to the streaming kernel with them."""
    x, w = rnd(M, K, seed=M, dtype=torch.bfloat16), rnd(N, K, seed=K, scale=0.1, dtype=torch.bfloat16)
    part = Linear(K, N, Precision.of("bfloat16"))
    part.load(w)
    y = part(x, torch.float32, allow_partials=True)
    check(y if y.dim() == 3 else y[None], x, w, K, y.shape[0] if y.dim() == 3 else 1)
