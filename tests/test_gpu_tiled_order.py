"""The tiled product's order of tiles (slices, bands of 1,024 tokens, columns): every tile once, at sizes around a band's end, with and
without slices of the inner dimension."""
import pytest
import torch
import torch.nn.functional as F

from alice_llm_amd.hip import ops
from test_gpu_kernels import rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"


def product(x, w, n_out, epi=ops.EPI_NONE, split=1):
    M, K = x.shape
    y = torch.full(((split,) if split > 1 else ()) + (M, n_out), float("nan"), dtype=torch.float32, device=DEV)
    ops.linear(x, w, y, n_out=n_out, k_in=K, layout=ops.LAYOUT_FRAG16, epilogue=epi, split_k=split, full_precision=False, variant=ops.LINEAR_AUTO)
    return y


@pytest.mark.parametrize("M", [66, 1023, 1024, 1025, 1153, 2049, 4500])
@pytest.mark.parametrize("N,K", [(16, 64), (272, 96), (2304, 160), (4112, 64)])
def test_every_tile_of_every_band_and_slice(M, N, K):
    x, w = rnd(M, K, seed=M, dtype=torch.bfloat16), rnd(N, K, seed=N, scale=0.1, dtype=torch.bfloat16)
    frag, ref = ops.to_frag16(w), x.double() @ w.double().T
    # products of bfloat16 numbers are exact in 32 bits: K additions of at most 2^-23 of all products' sizes
    tol = (x.double().abs() @ w.double().abs().T) * K * 2.0 ** -23
    whole = product(x, frag, N)
    assert ((whole.double() - ref).abs() <= tol).all()
    for split in (2, 3, 5):
        if split <= K // 32:
            assert ((product(x, frag, N, split=split).double().sum(0) - ref).abs() <= tol).all()
    for n in (min(M, 130), max(M - 70, 65)):                     # a token's sums do not hang on the others
        assert torch.equal(product(x[:n].contiguous(), frag, N), whole[:n])


@pytest.mark.parametrize("M", [1025, 3000])
@pytest.mark.parametrize("N", [32, 1168])
def test_every_tile_of_a_gated_product(M, N):
    K = 96
    x, w = rnd(M, K, seed=M, dtype=torch.bfloat16), rnd(2 * N, K, seed=N, scale=0.1, dtype=torch.bfloat16)
    ref = x.double() @ w.double().T
    got = product(x, ops.to_frag16(w), N, ops.EPI_GEGLU)
    # the fast tanh is good to 1e-6, the sums to K 2^-23 of about 10 K^1/2
    assert ((got.double() - F.gelu(ref[:, :N], approximate="tanh") * ref[:, N:]).abs() <= 1e-3 * (1 + ref[:, :N].abs() * ref[:, N:].abs())).all()
