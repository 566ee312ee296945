"""What the matrix recurrences take from the projection's rows, and the norm behind their read-out, at the edges of the
kernels: by tokens, by sequences and channel by channel, against each other and a 64-bit reference."""
import types

import pytest
import torch
import torch.nn.functional as F

from alice_llm_amd.hip import ops
from helpers import max_err

pytestmark = pytest.mark.gpu
DEV = "cuda"
FORMS = (ops.CONV_BY_TOKENS, ops.CONV_BY_SEQUENCES, ops.CONV_BY_CHANNELS)
LENS = [[1], [3, 0, 1, 2], [9, 1, 8], [17, 16]]              # around the tile of 8 tokens and pieces shorter than the taps


def rnd(*shape, seed=0, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


def step_of(lens, slots):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    i32 = dict(dtype=torch.int32, device=DEV)
    return types.SimpleNamespace(cu_seqlens=torch.tensor(cu, **i32), slots=torch.tensor(slots, **i32), n_seqs=len(lens), max_new=max(lens),
                                 seq_of_token=torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).to(torch.int32).to(DEV))


def conv_reference(x, w, b, state, lens, slots):
    """silu of the convolution in 64 bits, and the state behind the step."""
    K, outs, at, after = w.shape[1] - 1, [], 0, state.clone()
    for n, s in zip(lens, slots):
        full = torch.cat([state[s].T, x[at:at + n]]).double()
        y = sum(full[j:j + n] * w[:, j].double() for j in range(K + 1)) + (0.0 if b is None else b.double())
        outs.append(F.silu(y))
        after[s] = full[full.shape[0] - K:].T.float()
        at += n
    return torch.cat(outs), after


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("C,taps,col0,H", [(4, 2, 0, 1), (512, 3, 4, 3), (516, 4, 8, 130), (1028, 4, 0, 64)])
def test_state_space_enters(C, taps, col0, H, lens):
    T, row_w, slots = sum(lens), (col0 + C + H + 3) // 4 * 4, [5, 0, 3, 1][:len(lens)]
    x, w, b = rnd(T, row_w, seed=1), rnd(C, taps, seed=2, scale=0.6), rnd(C, seed=3)
    dt_bias, a_log, state = rnd(H, seed=4), rnd(H, seed=5, scale=0.5), rnd(6, C, taps - 1, seed=6)
    ref, after = conv_reference(x[:, col0:col0 + C], w, b, state, lens, slots)
    dt = F.softplus(x[:, col0 + C:col0 + C + H].double() + dt_bias.double())
    log = -torch.exp(a_log.double()) * dt
    got = []
    for form in FORMS:
        for as_log in (False, True):
            st, out = state.to(DEV), torch.empty(T, C, device=DEV)
            step, decay = torch.empty(T, H, device=DEV), torch.empty(T, H, device=DEV)
            ops.ssm_enter(x.to(DEV), col0, w.to(DEV), b.to(DEV), st, out, step_of(lens, slots), col0 + C, dt_bias.to(DEV), a_log.to(DEV),
                          step, decay, as_log=as_log, form=form)
            assert max_err(out, ref) < 1e-5 and torch.equal(st.cpu(), after), form
            # a handful of roundings and two ulps a function, relative to numbers of this size
            assert max_err(step, dt) < 1e-6 * float(dt.max()) and max_err(decay, log if as_log else log.exp()) < 2e-6 * max(1.0, float(log.abs().max()))
            got.append(out.cpu())
    assert all(torch.equal(g, got[0]) for g in got)           # the same products in the same order


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("G,H,d,dv,taps,low", [(1, 1, 4, 4, 2, torch.float32), (3, 6, 64, 32, 4, torch.bfloat16), (2, 2, 256, 128, 3, torch.bfloat16),
                                              (2, 4, 24, 12, 4, torch.float32), (5, 5, 128, 128, 4, torch.bfloat16), (1, 2, 6, 3, 4, torch.bfloat16)])
def test_delta_rule_enters(G, H, d, dv, taps, low, lens):
    C, n0, n1, eps, q_scale = 2 * G * d + H * dv, 5, 9, 1e-6, d ** -0.5
    T, row_w, slots = sum(lens), (C + H + n0 + n1 + 3) // 4 * 4, [5, 0, 3, 1][:len(lens)]
    x, w, state = rnd(T, row_w, seed=1), rnd(C, taps, seed=2, scale=0.6), rnd(6, C, taps - 1, seed=6)
    ref, after = conv_reference(x[:, :C], w, None, state, lens, slots)
    heads = ref[:, :2 * G * d].reshape(T, 2, G, d)
    heads = heads / torch.sqrt(heads.pow(2).sum(-1, keepdim=True) + eps)
    heads[:, 0] *= q_scale
    ref = torch.cat([heads.reshape(T, 2 * G * d), ref[:, 2 * G * d:]], 1)
    for form in FORMS:
        st, out, beta = state.to(DEV), torch.empty(T, C, device=DEV), torch.empty(T, H, device=DEV)
        a, g = torch.empty(T, n0, dtype=low, device=DEV), torch.empty(T, n1, dtype=low, device=DEV)
        ops.delta_enter(x.to(DEV), w.to(DEV), st, out, step_of(lens, slots), C, beta, C + H, a, g, qk_heads=G, head_dim=d, unit_eps=eps,
                        q_scale=q_scale, form=form)
        assert max_err(out, ref) < 1e-5 and torch.equal(st.cpu(), after), form
        assert max_err(beta, torch.sigmoid(x[:, C:C + H].double())) < 1e-6
        assert torch.equal(a.cpu(), x[:, C + H:C + H + n0].to(low)) and torch.equal(g.cpu(), x[:, C + H + n0:C + H + n0 + n1].to(low))


@pytest.mark.parametrize("T,H,d", [(1, 1, 1), (3, 5, 6), (7, 4, 64), (2, 3, 128)])
def test_delta_decays(T, H, d):
    z, dt_bias, a_log = rnd(T, H * d, seed=1, scale=3.0), rnd(H * d, seed=2), rnd(H, seed=3, scale=0.5)
    log = -torch.exp(a_log.double()).repeat_interleave(d) * F.softplus(z.double() + dt_bias.double())
    for as_log in (False, True):
        out = z.to(DEV)
        ops.delta_decay(out, dt_bias.to(DEV), a_log.to(DEV), heads=H, head_dim=d, as_log=as_log)
        assert max_err(out, log if as_log else log.exp()) < 2e-6 * max(1.0, float(log.abs().max()))


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("gate_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,n,parts", [(1, 4, 1), (3, 4, 5), (9, 128, 3), (5, 132, 1), (2, 512, 2), (3, 516, 1), (5, 1024, 1), (2, 1028, 1),
                                       (129, 1536, 2), (3, 4096, 1), (257, 4096, 1), (2, 4100, 1)])
def test_norm_and_gate_in_registers(T, n, parts, gate_dtype, out_dtype):
    width, eps = n * parts, 1e-5
    x, gate = rnd(T, width, seed=1, scale=3.0), rnd(T, width + 8, seed=2, scale=2.0).to(gate_dtype)
    g = gate.double()[:, 4:4 + width]
    for shared, act in ((False, "silu"), (True, "sigmoid"), (False, None)):
        w = rnd(n if shared else width, seed=3).abs() + 0.5
        y = (x.double() * F.silu(g) if act == "silu" else x.double()).view(T, parts, n)
        y = y / torch.sqrt(y.pow(2).mean(-1, keepdim=True) + eps) * (w.double() if shared else w.double().view(parts, n))
        y = y.reshape(T, width) * (torch.sigmoid(g) if act == "sigmoid" else 1.0)
        out = torch.empty(T, width, dtype=out_dtype, device=DEV)
        ops.norm_gate(x.to(DEV), w.to(DEV), out, parts=parts, eps=eps, weight_shared=shared, gate=None if act is None else gate.to(DEV),
                      gate_col=4, gate_act=act)
        # bfloat16: half a unit of the last of 8 bits of the largest number
        assert max_err(out, y) < (1e-5 if out_dtype == torch.float32 else 2 ** -8) * max(1.0, float(y.abs().max())), (shared, act)
