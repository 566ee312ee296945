"""The add and norm of few rows, four elements a thread: row lengths at the edges of its blocks, partial sums around what it
holds in registers, and addresses that it does not take (the kernel of one element at a time), against 64 bits."""
import pytest
import torch

from alice_llm_amd.hip import ops
from plain import gemma2_plain as P

pytestmark = pytest.mark.gpu
DEV = "cuda"
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def rnd(*shape, seed=0, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def close(got, ref, atol, rtol=0.0):
    err = (got.double() - ref.double()).abs()
    assert (err <= atol + rtol * ref.double().abs()).all(), f"max err {err.max().item():.3e}"


@pytest.mark.parametrize("H", [4, 252, 256, 260, 2300, 2304, 4096, 4100, 8188, 8192, 8196])
@pytest.mark.parametrize("S", [1, 4, 5, 8, 9, 17])
@pytest.mark.parametrize("wdt,odt", [("bfloat16", "bfloat16"), ("float32", "float32")])
def test_few_rows(H, S, wdt, odt):
    T = 3
    x0 = rnd(T, H, seed=2, scale=3.0)
    br = rnd(S, T, H, seed=3, scale=0.5) if S > 1 else rnd(T, H, seed=3, scale=0.5)
    wp, wq = rnd(H, seed=4, scale=0.1, dtype=DT[wdt]), rnd(H, seed=5, scale=0.1, dtype=DT[wdt])
    tol = 2e-6 if odt == "float32" else 2 ** -8
    full = odt == "float32"
    want = x0.double() + P.rms_norm(br.double().sum(0) if S > 1 else br.double(), wp.double(), 1e-6)
    x, out = x0.clone(), torch.full((T, H), float("nan"), dtype=DT[odt], device=DEV)
    ops.add_norm(x, br, wp, wq, out, eps_post=1e-6, eps_pre=1e-5, off_post=1.0, off_pre=1.0, n_partials=S, full_precision=full)
    close(x, want, 1e-5)
    close(out, P.rms_norm(want, wq.double(), 1e-5), tol * 4, tol)
    # the same operands one element further on: no multiple of 16 bytes
    def moved(t):
        u = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
        return u.copy_(t)
    x2, out2 = moved(x0), moved(out)
    ops.add_norm(x2, moved(br), moved(wp), moved(wq), out2, eps_post=1e-6, eps_pre=1e-5, off_post=1.0, off_pre=1.0, n_partials=S,
                 full_precision=full)
    close(x2, want, 1e-5)
    close(out2, P.rms_norm(want, wq.double(), 1e-5), tol * 4, tol)


@pytest.mark.parametrize("H", [4, 260, 4096, 4100, 8192])
def test_mean_and_bias_of_few_rows(H):
    T = 5
    x0, br = rnd(T, H, seed=2, scale=3.0) + 1.5, rnd(2, T, H, seed=3)
    w, b = rnd(H, seed=4), rnd(H, seed=5)
    x, out = x0.clone(), torch.full((T, H), float("nan"), device=DEV)
    ops.add_norm(x, br, None, w, out, eps_pre=1e-5, n_partials=2, full_precision=True, b_pre=b)
    want = x0.double() + br.double().sum(0)
    close(x, want, 1e-5)
    close(out, torch.nn.functional.layer_norm(want, (H,), w.double(), b.double(), 1e-5), 2e-5)
    rows = torch.tensor([4, 0, 4], dtype=torch.int32, device=DEV)
    out = torch.full((3, H), float("nan"), device=DEV)
    ops.add_norm(x0, None, None, w, out, eps_pre=1e-5, rows=rows, full_precision=True, b_pre=b)
    close(out, torch.nn.functional.layer_norm(x0.double()[rows.long()], (H,), w.double(), b.double(), 1e-5), 2e-5)
