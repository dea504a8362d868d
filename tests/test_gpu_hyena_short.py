"""The Hyena operator on short rows in one launch (csrc/hyena.hip hyena_short_kernel) against the oracle in fp64: numbers of positions on both sides of the 32
segments' edges, and a prefix's state and history carried in.  Tolerances: as the three launches' (test_gpu_kernels.test_hyena_prefill_matches_oracle)."""
import pytest
import torch

from oracle import stripedhyena_ref as R
from test_gpu_kernels import assert_close_bf16, bf, gen, hyena_params, ops, run_hyena  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,D,H", [(1, 1, 128, 1), (2, 2, 128, 1), (1, 31, 256, 2), (3, 32, 128, 1), (1, 33, 128, 1), (2, 95, 256, 2), (1, 97, 128, 1), (1, 161, 4096, 32),
                                     (1, 992, 128, 1), (1, 993, 128, 1), (1, 1023, 256, 2)])
def test_short_rows(ops, B, T, D, H):
    prm = hyena_params(D, T)
    z = bf(torch.randn(B, T, 3 * D, generator=gen(T + 1)))
    calls = []
    real = ops._t
    ops._t = lambda name: (calls.append(name), real(name))[1]
    try:
        y, st = run_hyena(ops, z, prm, H, want_state=True)
    finally:
        del ops._t
    assert calls == ["hyena_short"]
    ry, rst = R.op_hyena(z, *prm, H)
    rl2 = 2e-3 if B * T * D >= 2048 else 2.0 ** -8               # (few values: one of them may be most of the norm, and half an ulp is 2^-8 of it)
    assert_close_bf16(y, ry, rl2)
    assert (st.cpu().to(torch.complex128) - rst).abs().max() <= 2e-5 * rst.abs().max()
    y3, st3 = run_hyena(ops, z, prm, H, want_state=True, seg_len=64)                # the three launches
    assert_close_bf16(y, y3.float().cpu(), rl2)
    assert (st - st3).abs().max() <= 2e-5 * st3.abs().max()
    assert torch.equal(run_hyena(ops, z, prm, H)[0], y)                             # without a state
    if T >= 3:                                                                      # behind a prefix, in one batch
        cut = T // 3 + 1
        _, s1 = run_hyena(ops, z[:, :cut].contiguous(), prm, H, want_state=True)
        halo = torch.cat([z.new_zeros(B, 2, 3 * D), z[:, :cut]], 1)[:, -2:].contiguous()
        y2, s2 = run_hyena(ops, z[:, cut:].contiguous(), prm, H, want_state=True, z_halo=halo, s0=s1)
        assert_close_bf16(y2, ry[:, cut:], rl2)
        assert (s2.cpu().to(torch.complex128) - rst).abs().max() <= 2e-5 * rst.abs().max()


@pytest.mark.parametrize("T,lo,hi", [(1, 0, 1), (40, 0, 3), (201, 150, 201), (201, 77, 80), (640, 100, 400)])
def test_masked_positions(ops, T, lo, hi):
    """Padded positions lo .. hi - 1 of the second row, against the three launches; where nothing is padded, and in front of a padded tail, the unmasked bits."""
    prm, z = hyena_params(128, 5), bf(torch.randn(2, T, 384, generator=gen(6)))
    mask = torch.ones(2, T, dtype=torch.bool)
    mask[1, lo:hi] = False
    y, st = run_hyena(ops, z, prm, 1, want_state=True, mask=mask)
    y3, st3 = run_hyena(ops, z, prm, 1, want_state=True, mask=mask, seg_len=32)
    plain = run_hyena(ops, z, prm, 1)[0]
    assert_close_bf16(y, y3.float().cpu(), 2e-3 if T >= 40 else 2.0 ** -8)
    assert (st - st3).abs().max() <= 2e-5 * st3.abs().max()
    assert torch.equal(y[0], plain[0]) and torch.equal(y[1, :lo], plain[1, :lo]) and bool((y[1, lo:hi] == 0).all())


def test_longer_rows_take_the_three_launches(ops):
    """From 1,024 positions on, where a row's bits are the same in every batch."""
    names = []
    for B, T in ((1, 1024), (2, 512), (1, 1025)):
        prm, z = hyena_params(128, 3), bf(torch.randn(B, T, 384, generator=gen(4)))
        real = ops._t
        ops._t = lambda name: (names.append(name), real(name))[1]
        try:
            both = run_hyena(ops, z, prm, 1)[0]
            assert torch.equal(run_hyena(ops, torch.cat([z, z]), prm, 1)[0][:B], both)
        finally:
            del ops._t
    assert "hyena_short" not in names
    prm, z = hyena_params(128, 3), bf(torch.randn(1, 1025, 384, generator=gen(4)))
    y, _ = run_hyena(ops, z, prm, 1)
    assert_close_bf16(y, R.op_hyena(z, *prm, 1)[0])
    args = [z.cuda()] + [t.cuda() for t in prm] + [y]
    p = [t.data_ptr() for t in args]
    assert ops.lib.evo_hyena_short(p[0], None, p[1], p[2], p[3], p[4], p[5], None, None, p[6], None, 1, 1025, 128, 1, None) == -1
    assert ops.lib.evo_hyena_short(p[0] + 8, None, p[1], p[2], p[3], p[4], p[5], None, None, p[6], None, 1, 16, 128, 1, None) == -1
