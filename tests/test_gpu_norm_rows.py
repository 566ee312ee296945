"""Residual add and norms of many rows: the widths between which the waves a row and the elements a lane change, and fragment order."""
import pytest
import torch

from alice_llm_amd.hip import ops
from plain import gemma2_plain as P
from test_gpu_kernels import DEV, acts_from_fragments, close, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [320, 333, 1040])
@pytest.mark.parametrize("H", [256, 1024, 1028, 2048, 2052, 2560, 2592, 3584, 3588, 4608, 4640, 8192])
def test_many_rows(T, H):
    x0, br = rnd(T, H, seed=2, scale=3.0), rnd(T, H, seed=3, scale=0.5)
    wp, wq = rnd(H, seed=4, scale=0.1, dtype=torch.bfloat16), rnd(H, seed=5, scale=0.1, dtype=torch.bfloat16)
    kw = dict(eps_post=1e-6, eps_pre=1e-5, off_post=1.0, off_pre=1.0, full_precision=False)
    xr = x0.double() + P.rms_norm(br.double(), wp.double(), 1e-6)
    x, row = x0.clone(), torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.add_norm(x, br, wp, wq, row, **kw)
    close(x, xr, 1e-5)
    close(row, P.rms_norm(xr, wq.double(), 1e-5), 2 ** -6, 2 ** -8)
    if H % 32 == 0:
        x, flat = x0.clone(), torch.full((-(-T // 16) * 16 * H,), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.add_norm(x, br, wp, wq, flat, out_layout=ops.LAYOUT_FRAG16, **kw)
        close(x, xr, 1e-5)
        assert torch.equal(acts_from_fragments(flat, T, H), row.cpu())
        assert int(flat.isnan().sum()) == (-T % 16) * H         # rows past the end stay as they were


# the widths' other forms: 32-bit rows with sums over slices, the centred norm with a bias over both orders of the output, the add alone
@pytest.mark.parametrize("H", [256, 1024, 1028, 2048, 2052, 2560, 2592, 3584, 3588, 4608, 4640, 8192])
@pytest.mark.parametrize("form", ["f32", "centred", "add"])
def test_many_rows_other_forms(H, form):
    T, n = 333, 3
    x0, br = rnd(T, H, seed=2, scale=3.0), rnd(n, T, H, seed=3, scale=0.5)
    wp, wq, b = rnd(H, seed=4, scale=0.1), rnd(H, seed=5, scale=0.1), rnd(H, seed=6, scale=0.1)
    xr = x0.double() + P.rms_norm(br.double().sum(0), wp.double(), 1e-6)
    kw = dict(eps_post=1e-6, off_post=1.0, eps_pre=1e-5, off_pre=1.0, n_partials=n)
    x = x0.clone()
    if form == "add":
        ops.add_norm(x, br, wp, None, None, full_precision=True, **kw)
    elif form == "f32":
        out = torch.full((T, H), float("nan"), device=DEV)
        ops.add_norm(x, br, wp, wq, out, full_precision=True, **kw)
        close(out, P.rms_norm(xr, wq.double(), 1e-5), 1e-5, 2e-6)   # (32-bit sums of up to 8,192 squares, and the row's own 1e-5 of up to 15)
    else:
        out = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.add_norm(x, br, wp, wq, out, full_precision=False, b_pre=b, **kw)
        ref = torch.nn.functional.layer_norm(xr, (H,), None, None, 1e-5) * (1 + wq.double()) + b.double()
        close(out, ref, 1e-4, 2 ** -8)                       # one rounding to bfloat16
        if H % 32 == 0:
            y, flat = x0.clone(), torch.full((-(-T // 16) * 16 * H,), float("nan"), dtype=torch.bfloat16, device=DEV)
            ops.add_norm(y, br, wp, wq, flat, full_precision=False, b_pre=b, out_layout=ops.LAYOUT_FRAG16, **kw)
            assert torch.equal(acts_from_fragments(flat, T, H), out.cpu()) and torch.equal(x, y)
    close(x, xr, 1e-5, 1e-6)
