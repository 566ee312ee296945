"""The gate functions of the products' epilogues by themselves: gates of known numbers, an up half of ones."""
import pytest
import torch

from alice_llm_amd.hip import ops
from test_gpu_kernels import acts_from_fragments, acts_to_fragments

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(M, N, K):
    """Row m's products are z[m] (16 bits of it, as two bfloat16 parts, so that every sum is exact) and 1."""
    z = torch.linspace(-9, 9, M, device=DEV)
    hi = z.to(torch.bfloat16)
    lo = (z - hi.float()).to(torch.bfloat16)
    x = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
    x[:, 0], x[:, 1], x[:, 2] = hi, lo, 1.0
    one, gated = torch.zeros(N, K, dtype=torch.bfloat16, device=DEV), torch.zeros(2 * N, K, dtype=torch.bfloat16, device=DEV)
    one[:, :2], gated[:N, :2], gated[N:, 2] = 1.0, 1.0, 1.0
    return hi.float() + lo.float(), x, one, gated


# rows of tokens and weights: the plain kernel; fragments: the streaming kernel, the tiled one, and (in bfloat16) the large tiles
@pytest.mark.parametrize("layout,M,dtype,variant", [
    (ops.LAYOUT_ROW, 40, torch.float32, ops.LINEAR_AUTO), (ops.LAYOUT_ROW, 1000, torch.float32, ops.LINEAR_AUTO),
    (ops.LAYOUT_FRAG16, 64, torch.float32, ops.LINEAR_AUTO), (ops.LAYOUT_FRAG16, 4099, torch.float32, ops.LINEAR_AUTO),
    (ops.LAYOUT_FRAG16, 4099, torch.bfloat16, ops.LINEAR_LARGE_256)])
def test_silu_is_one_function(layout, M, dtype, variant):
    """A gate of silu(z) times 1 has the bits of the function of one element, silu(z): one division, rounded once."""
    N, K = 32, 128
    z, x, one, gated = operands(M, N, K)
    if layout == ops.LAYOUT_FRAG16:
        one, gated = ops.to_frag16(one), ops.to_frag16(gated)
    frag = variant != ops.LINEAR_AUTO
    kw = dict(n_out=N, k_in=K, layout=layout, full_precision=False, rows=M)
    alone, gate = torch.empty(M, N, dtype=dtype, device=DEV), torch.empty(M, N, dtype=dtype, device=DEV)
    ops.linear(x, one, alone, epilogue=ops.EPI_SOFTCAP, epi_param=ops.UNARY_SILU, **kw)
    ops.linear(acts_to_fragments(x) if frag else x, gated, gate, epilogue=ops.EPI_GEGLU, epi_param=ops.GATED_SILU, variant=variant,
               x_layout=ops.LAYOUT_FRAG16 if frag else ops.LAYOUT_ROW, **kw)
    assert torch.equal(gate, alone)
    ref = torch.nn.functional.silu(z.double())[:, None]
    # the exponential's argument is off by 2^-24 of up to 13 (base 2), its value by one unit more; the division and the sum round
    assert ((gate.double() - ref).abs() <= (2 ** -8 if dtype == torch.bfloat16 else 2e-6) * ref.abs()).all()


@pytest.mark.parametrize("M", [64, 4099])
def test_gelu(M):
    N, K = 32, 128
    z, x, _, gated = operands(M, N, K)
    y = torch.empty(M, N, device=DEV)
    ops.linear(x, ops.to_frag16(gated), y, n_out=N, k_in=K, layout=ops.LAYOUT_FRAG16, epilogue=ops.EPI_GEGLU, full_precision=False)
    ref = torch.nn.functional.gelu(z.double(), approximate="tanh")[:, None]
    # results above 1e-6 have an exponent (base 2) of up to 31, off by 2.5 * 2^-24 of itself: 3.2e-6 of the result
    big = ref.abs() > 1e-6
    assert ((y.double() - ref).abs() <= torch.where(big, 4e-6 * ref.abs(), torch.full_like(ref, 1e-11))).all()
