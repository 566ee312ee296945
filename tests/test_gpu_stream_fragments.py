"""The stream itself, without a norm, in the matrix products' fragment order: the same numbers as in rows."""
import pytest
import torch

from alice_llm_amd.parts.base import FragmentActs, Precision
from alice_llm_amd.parts.linear import Linear
from alice_llm_amd.parts.norm import RMSNorm
from alice_llm_amd.parts.stream import ResidualStream
from test_gpu_kernels import acts_from_fragments, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,H", [(1, 64), (15, 2304), (17, 96), (32, 2048), (65, 2048), (319, 160), (320, 256), (333, 2048), (700, 4128)])
@pytest.mark.parametrize("slices,post", [(0, False), (1, False), (1, True), (3, True)])
def test_the_stream_without_a_norm_in_fragment_order(T, H, slices, post):
    precision = Precision.of("bfloat16")
    norm = None
    if post:
        norm = RMSNorm(precision, dim=H, eps=1e-6, weight_offset=1.0)
        norm.assign("weight", rnd(H, seed=3, scale=0.1, dtype=torch.bfloat16))
    outs, streams = [], []
    for fragments in (False, True):
        s = ResidualStream(rnd(T, H, seed=1), precision)
        if slices:
            s.push(rnd(*((slices,) if slices > 1 else ()), T, H, seed=2), norm)
        outs.append(s.normed(None, fragments=fragments))
        streams.append(s)
    assert isinstance(outs[1], FragmentActs) and outs[1].shape == (T, H)
    assert torch.equal(acts_from_fragments(outs[1].data, T, H), outs[0].cpu())
    assert torch.equal(streams[0].x, streams[1].x) and streams[1]._branch is None


@pytest.mark.parametrize("T", [33, 64])
def test_rows_where_the_order_of_the_sums_would_change(T):
    s = ResidualStream(rnd(T, 256, seed=1), Precision.of("bfloat16"))
    s.push(rnd(T, 256, seed=2))
    out = s.normed(None, fragments=True)
    assert torch.equal(out, s.x.to(torch.bfloat16))


# outputs and widths of a delta layer's projection (tiled from one token on if it were given fragment order), and streaming ones; GeGLU
# (from 448 tokens on fragment order has a kernel more, which would like other slices)
@pytest.mark.parametrize("T", [1, 8, 16, 32, 33, 64, 65, 130, 447, 448, 700, 2048])
@pytest.mark.parametrize("N,H", [(12576, 4096), (12224, 4096), (2304, 4128), (12576, 2048), (2560, 1024), (2304, 2304)])
def test_the_product_behind_the_stream_without_a_norm(T, N, H):
    """The same bits whether the consumer says that it reads fragment order or not."""
    precision = Precision.of("bfloat16")
    part = Linear(H, N, precision)
    part.load(rnd(N, H, seed=5, scale=0.1, dtype=torch.bfloat16))
    x, branch = rnd(T, H, seed=1), rnd(T, H, seed=2)
    outs = []
    for fragments in (False, True):
        s = ResidualStream(x.clone(), precision)
        s.push(branch)
        acts = s.normed(None, fragments=fragments)
        outs.append([part(acts, torch.float32, allow_partials=True), part(acts, torch.float32), part(acts, torch.bfloat16)])
    assert all(torch.equal(a, b) for a, b in zip(*outs))
