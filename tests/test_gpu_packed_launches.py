"""GPU: unequal sequences in one launch (evo_hyena_ct_packed, evo_attn_fwd_packed_bf16) against a launch each, bit for bit where both run the same tiles, and many copies
in one launch (evo_copy_rows).  Rows between the sequences hold NaN: nothing of them may reach a result."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ops():
    from evo_amd.ops import default_ops
    return default_ops()


def _places(lens):
    first, M = [], 0
    for m in lens:
        first.append(M)
        M += (m + 63) // 64 * 64
    return first, (M + 255) // 256 * 256


# lengths at the edges of 64-row places, of 512-step tiles and of the workgroups that share a group of channels (one at 32 heads, eight at four)
@pytest.mark.parametrize("H,lens", [(4, [33, 64, 65, 1, 127, 512, 513, 40, 1030]), (4, [70]), (32, [511, 33, 512, 1024, 8, 1025])])
def test_hyena(H, lens):
    from evo_amd.hyena_tables import mfma_operand_table
    ops, D = _ops(), H * 128
    g = torch.Generator().manual_seed(sum(lens))
    mag, ang = 1.0 - 10.0 ** (-5.0 + 4.0 * torch.rand(D, 8, generator=g)), (torch.rand(D, 8, generator=g) * 2 - 1) * math.pi
    poles = torch.stack([mag * torch.cos(ang), mag * torch.sin(ang)], -1).float().contiguous().to(DEV)
    res = (torch.randn(D, 8, 2, generator=g) * 0.25).float().contiguous().to(DEV)
    table = mfma_operand_table(poles, res, (torch.randn(D, generator=g) * 0.5).bfloat16().to(DEV))
    fw, fb = (torch.randn(3 * D, 3, generator=g) * 0.3).bfloat16().to(DEV), (torch.randn(3 * D, generator=g) * 0.1).bfloat16().to(DEV)
    first, M = _places(lens)
    zt = torch.full((M // 256, 3 * D, 256), float("nan"), device=DEV, dtype=torch.bfloat16)
    for f, m in zip(first, lens):
        at = torch.arange(f, f + m, device=DEV)
        zt[at // 256, :, at % 256] = torch.randn(m, 3 * D, generator=g).bfloat16().to(DEV)
    seqs = torch.tensor(list(zip(first, lens)), dtype=torch.int32)
    state, keep = torch.empty(len(lens), D, 8, dtype=torch.complex64, device=DEV), torch.full((1,), 7.0, device=DEV, dtype=torch.bfloat16)
    y = keep.expand(ops.yblk_empty(M, D, DEV).shape).contiguous()
    ops.hyena_ct_packed(zt, fw, fb, table, H, seqs.to(DEV), seqs, poles, y, state)
    want, alone = y.new_full(y.shape, 7.0), torch.empty_like(state)
    for n, (f, m) in enumerate(zip(first, lens)):
        ops.hyena_ct(zt, 1, m, fw, fb, table, H, want_state=True, poles=poles, y_blk=want, y_row0=f, at=f, s_out=alone[n:n + 1])
    assert torch.equal(y, want) and torch.equal(torch.view_as_real(state), torch.view_as_real(alone)) and bool(torch.isfinite(y).all())
    for bad in ([[0, M + 1]], [[4, 8]], [[-8, 8]], [[0, 0]]):        # out of the tensor, off a multiple of 8, empty
        t = torch.tensor(bad, dtype=torch.int32)
        with pytest.raises(Exception):
            ops.hyena_ct_packed(zt, fw, fb, table, H, t.to(DEV), t, poles, y, state[:1].contiguous())


# lengths at the edges of 64 keys, 128 and 256 queries
@pytest.mark.parametrize("H,lens", [(4, [1, 33, 64, 65, 127, 128, 129, 255, 256, 257, 700]), (5, [300, 40]), (32, [1030, 129, 513])])
@pytest.mark.parametrize("prescaled", [False, True])
def test_attention(H, lens, prescaled, monkeypatch):
    ops = _ops()
    monkeypatch.setattr(ops, "attn_w64_from", 0, raising=False)           # (alone, a short prompt takes the other kernel: test_gpu_few_launches.py)
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    first, M = _places(lens)
    qkv = torch.full((M, 3, H, 128), float("nan"), device=DEV, dtype=torch.bfloat16)
    for f, m in zip(first, lens):
        qkv[f:f + m] = torch.randn(m, 3, H, 128, device=DEV, generator=g).bfloat16()
    if prescaled:
        qkv[:, 0] = (qkv[:, 0].float() * ops.attn_q_scale(128)).bfloat16()
    blocks, valid = ops.packed_blocks(first, lens, M)
    out = torch.full((M, H * 128), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.attention_packed(qkv[:, 0], qkv[:, 1], qkv[:, 2], blocks.to(DEV), blocks, valid.to(DEV), out, prescaled=prescaled)
    inside = torch.zeros(M, dtype=torch.bool, device=DEV)
    for f, m in zip(first, lens):
        inside[f:f + m] = True
        q, k, v = (qkv[f:f + m, i][None] for i in range(3))
        alone = ops.attention(q, k, v, 0, prescaled=prescaled)[0].reshape(m, H * 128)
        if m > 128:                                                   # the same kernel
            assert torch.equal(out[f:f + m], alone), m
        else:                                                         # (two bf16 kernels: each within 2^-8 of the result's row and 2e-3 for the weights' rounding)
            assert ((out[f:f + m].double() - alone.double()).norm() / alone.double().norm()).item() < 1e-2, m
    assert bool((out[~inside] == 7.0).all())
    for bad in ([[0, M + 1, 0, 0]], [[32, 300, 0, 0]], [[0, 300, 100, 0]], [[0, 300, -256, 0]]):
        t = torch.tensor(bad, dtype=torch.int32)
        with pytest.raises(Exception):
            ops.attention_packed(qkv[:, 0], qkv[:, 1], qkv[:, 2], t.to(DEV), t, valid.to(DEV), out)


# a sequence on each kernel, at the edges between them (the line between 8 waves and 64 rows a wave lowered to 640 keys, and where it is)
@pytest.mark.parametrize("H,lens,first", [(4, [1, 128, 129, 255, 256, 257, 639, 640, 641, 64, 1100], 640), (5, [128, 40], None), (32, [1030, 129, 513], None),
                                          (4, [3499, 100, 3500, 3501, 1300], None)])
@pytest.mark.parametrize("prescaled", [False, True])
def test_attention_has_the_bits_of_each_sequence_alone(H, lens, first, prescaled, monkeypatch):
    ops = _ops()
    if first is not None:
        monkeypatch.setattr(ops, "attn_w64_from", first, raising=False)
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    at, M = _places(lens)
    qkv = torch.full((M, 3, H, 128), float("nan"), device=DEV, dtype=torch.bfloat16)
    for f, m in zip(at, lens):
        qkv[f:f + m] = torch.randn(m, 3, H, 128, device=DEV, generator=g).bfloat16()
    blocks, valid = ops.packed_blocks(at, lens, M)
    assert sorted(set(blocks[:, 3].tolist())) == sorted({0 if m <= 128 else 1 if m < (first or 3500) else 2 for m in lens})
    out = torch.full((M, H * 128), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.attention_packed(qkv[:, 0], qkv[:, 1], qkv[:, 2], blocks.to(DEV), blocks, valid.to(DEV), out, prescaled=prescaled)
    inside = torch.zeros(M, dtype=torch.bool, device=DEV)
    for f, m in zip(at, lens):
        inside[f:f + m] = True
        q, k, v = (qkv[f:f + m, i][None] for i in range(3))
        assert torch.equal(out[f:f + m], ops.attention(q, k, v, 0, prescaled=prescaled)[0].reshape(m, H * 128)), m
    assert bool((out[~inside] == 7.0).all())
    for bad in ([0, 100, 1, 0], [0, 300, 0, 0], [0, 300, 128, 1], [0, 300, 512, 1], [0, 100, 0, 1], [0, 300, 100, 2], [0, M + 64, 0, 1], [32, 300, 0, 1], [0, 300, 0, 3]):
        t = torch.tensor([bad], dtype=torch.int32)
        with pytest.raises(Exception):
            ops.attention_packed(qkv[:, 0], qkv[:, 1], qkv[:, 2], t.to(DEV), t, valid.to(DEV), out)


def test_copies():
    """Dense pieces, rows at a pitch, one element, nothing, sizes off 16 bytes, more pieces than one launch takes; what lies beside them stays."""
    ops = _ops()
    g = torch.Generator().manual_seed(3)
    pairs, beside = [], []
    for rows, cols, pitch, dtype in [(1, 8, 8, torch.float32), (5, 4096, 6144, torch.bfloat16), (300, 64, 72, torch.float32), (7, 3, 3, torch.bfloat16), (4, 5, 9, torch.float32),
                                     (0, 8, 8, torch.float32), (1, 1 << 20, 1 << 20, torch.bfloat16)] + [(3, 16, 24, torch.float32)] * 130:
        src = torch.randn(rows, pitch, generator=g).to(dtype).to(DEV)[:, :cols]
        whole = torch.zeros(rows, pitch + 8, dtype=dtype, device=DEV)
        pairs.append((whole[:, :cols], src))
        beside.append(whole[:, cols:])
    z = torch.randn(6, 8, 2, generator=g).to(DEV)
    pairs.append((torch.zeros(6, 8, dtype=torch.complex64, device=DEV), torch.view_as_complex(z)))
    ops.copy_rows(pairs)
    assert all(torch.equal(d, s) for d, s in pairs) and not any(b.any() for b in beside)
    with pytest.raises(RuntimeError):
        ops.copy_rows([(torch.zeros(2, 8, device=DEV), torch.zeros(3, 8, device=DEV))])
