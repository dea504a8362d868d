"""Decayed linear attention token by token: the prompt kernel (eight tokens between barriers, state in registers up to 128 rows) does the decode
step's arithmetic in the decode step's order."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from evo_amd.ops import HipOps
    return HipOps()


# state rows: fewer than a thread's share, its edge, past it (state in LDS), the widest quad and the widest plain form; value columns: tiles of 32 (8)
# with and without remainders.  Lengths: none, one, a block, one more, several and a rest.
@pytest.mark.parametrize("dk,dv", [(5, 4), (32, 36), (100, 5), (128, 128), (129, 36), (200, 130), (1024, 32), (1100, 12)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("act", [0, 1])
def test_prompts_are_the_steps(ops, dt, dk, dv, act):
    H, lens, pad = 2, [1, 8, 0, 9, 27, 7], 3
    g = torch.Generator().manual_seed(dk)
    n, M, B = H * (2 * dk + dv), sum(lens), len(lens)
    z = torch.randn(M, n + pad, generator=g).to(dt).to(DEV)
    dec = torch.tensor([0.9, 1.0], device=DEV)
    cu = torch.tensor([0] + lens, dtype=torch.int64).cumsum(0).to(torch.int32).to(DEV)
    resume = torch.tensor([0, 1, 1, 0, 1, 0], dtype=torch.int32, device=DEV)
    first = torch.randn(B, H, dk, dv, generator=g).to(DEV)
    st, o = first.clone(), torch.zeros(M, H * dv, dtype=dt, device=DEV)
    f32 = int(dt == torch.float32)
    ops._call("evo_lightning_recurrent", z.data_ptr(), z.stride(0), o.data_ptr(), st.data_ptr(), dec.data_ptr(), cu.data_ptr(), resume.data_ptr(), B, H, dk, dv, act, f32)
    at = 0
    for b, L in enumerate(lens):
        s = first[b].clone() if int(resume[b]) else torch.zeros_like(first[b])
        for t in range(L):
            y = torch.empty(1, H * dv, dtype=dt, device=DEV)
            ops._call("evo_lightning_recurrent", z[at + t].data_ptr(), z.stride(0), y.data_ptr(), s.data_ptr(), dec.data_ptr(), None, None, 1, H, dk, dv, act, f32)
            assert torch.equal(o[at + t], y[0]), (b, t)
        assert torch.equal(st[b], s) or L == 0, b
        at += L
