"""Decayed linear attention of fp32 prompts in chunks of 32 tokens (csrc/lightning.hip lightning_f32_kernel): chunk edges, columns that don't fill a block, carried
states, decays of 0 and 1 and negative ones, values that are not finite, and the layouts that the token form keeps."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def run(z, H, dk, dv, decay, lens, state=None, resume=None, act=0):
    from evo_amd.ops import _stream, default_ops
    M = sum(lens)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0)], dtype=torch.int32, device="cuda")
    o = torch.full((M + 2, H * dv), 7.0, device="cuda")
    st = torch.full((len(lens), H, dk, dv), 1e6, device="cuda") if state is None else state.clone()
    assert default_ops().lib.evo_lightning_recurrent(z.data_ptr(), z.stride(0), o.data_ptr(), st.data_ptr(), decay.data_ptr(), cu.data_ptr(), None if resume is None else resume.data_ptr(),
                                       len(lens), H, dk, dv, act, 1, _stream()) == 0
    assert bool((o[M:] == 7).all())
    return o[:M], st


def want(z, H, dk, dv, decay, lens, state=None, resume=None):
    out, states, at = [], [], 0
    for b, n in enumerate(lens):
        x = z[at:at + n].double()
        q, k, v = x[:, :H * dk].view(n, H, dk), x[:, H * dk:2 * H * dk].view(n, H, dk), x[:, 2 * H * dk:H * (2 * dk + dv)].view(n, H, dv)
        S = state[b].double() if state is not None and resume[b] else torch.zeros(H, dk, dv, dtype=torch.float64, device="cuda")
        for t in range(n):
            S = decay.double()[:, None, None] * S + k[t][:, :, None] * v[t][:, None, :]
            out.append((S * q[t][:, :, None]).sum(1).reshape(-1))
        states.append(S)
        at += n
    return torch.stack(out), torch.stack(states)


@pytest.mark.parametrize("H,dk,dv,extra", [(5, 64, 64, 0), (3, 128, 128, 4), (2, 128, 36, 8), (1, 64, 4, 0), (2, 128, 64, 1), (2, 64, 33, 0)])
def test_chunks(H, dk, dv, extra):
    """(the last two: rows or columns that are no multiple of 16 bytes, token by token)  A sum of n fp32 terms is off by under sqrt(n) 2^-24 of its terms' norm; 128 rows and
    up to 130 tokens: 2e-6 of the result covers it tenfold."""
    lens = [1, 31, 32, 33, 64, 130, 3]
    g = torch.Generator(device="cuda").manual_seed(dk + dv)
    z = torch.randn(sum(lens), H * (2 * dk + dv) + extra, device="cuda", generator=g)
    decay = torch.tensor([0.0, 1.0, 0.97, -0.9, 0.5][:H] if H == 5 else [0.999, 0.3, 0.9][:H], device="cuda")
    state = torch.randn(len(lens), H, dk, dv, device="cuda", generator=g)
    resume = torch.tensor([1, 0, 1, 1, 0, 1, 1], dtype=torch.int32, device="cuda")
    o, st = run(z, H, dk, dv, decay, lens, state, resume)
    wo, ws = want(z, H, dk, dv, decay, lens, state, resume)
    assert ((o.double() - wo).norm() / wo.norm()).item() < 2e-6 and ((st.double() - ws).norm() / ws.norm()).item() < 2e-6
    assert bool(((o.double() - wo).norm(dim=1) < 1e-5 * wo.norm(dim=1)).all())
    o1, s1 = run(z, H, dk, dv, decay, lens)                       # from nothing, whatever the slot held
    w1, t1 = want(z, H, dk, dv, decay, lens)
    assert ((o1.double() - w1).norm() / w1.norm()).item() < 2e-6 and ((s1.double() - t1).norm() / t1.norm()).item() < 2e-6
    oa, sa = run(z, H, dk, dv, decay, lens, act=1)
    wa, ta = want(torch.nn.functional.silu(z.double()), H, dk, dv, decay, lens)
    assert ((oa.double() - wa).norm() / wa.norm()).item() < 4e-6 and ((sa.double() - ta).norm() / ta.norm()).item() < 4e-6


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_values_that_are_not_finite_reach_later_tokens_only(bad):
    H, dk, dv, lens, at = 2, 64, 64, [40, 40], 20
    g = torch.Generator(device="cuda").manual_seed(3)
    z = torch.randn(80, H * (2 * dk + dv), device="cuda", generator=g)
    decay = torch.tensor([0.9, 0.5], device="cuda")
    clean, _ = run(z, H, dk, dv, decay, lens)
    z[at, 2 * H * dk + 5] = bad                                   # column 5 of head 0's values
    o, st = run(z, H, dk, dv, decay, lens)
    hit = torch.zeros_like(o, dtype=torch.bool)
    hit[at:40, 5] = True
    assert not bool(torch.isfinite(o[hit]).any()) and bool(((o - clean)[~hit].abs() <= 1e-5 * (clean[~hit].abs() + 1)).all())
    assert not bool(torch.isfinite(st[0, 0, :, 5]).any()) and bool(torch.isfinite(st[1]).all()) and bool(torch.isfinite(st[0, 1]).all())
