"""Short inputs: the scoring tail as a dense layer and one kernel over its logits, and the modal Hyena operator on segments of 4 to 64 positions."""
import math
import pytest
import torch
from oracle import stripedhyena_ref as R
from test_gpu_kernels import DEV, assert_close_bf16, bf, gen, hyena_params, run_hyena

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from evo_amd.ops import HipOps
    return HipOps()


@pytest.mark.parametrize("M,K", [(5, 192), (64, 128), (65, 4096), (161, 4096), (1023, 256), (1024, 256), (4101, 256), (31, 96)])
def test_tail_matches_the_oracle(ops, M, K):
    """Widths the dense layer takes (K % 64 == 0) and one it does not.  One rounding of every logit: where the fp32 sum lies within its own error of a
    rounding boundary the logit is one bf16 step off, which moves a log-probability by that step and the entropy by its probability's share."""
    hid = bf(torch.randn(M, K, generator=gen(40)))
    emb = bf(torch.randn(512, K, generator=gen(41)) * (4.0 / math.sqrt(K)))
    tgt = torch.randint(0, 512, (M,), generator=gen(42))
    tgt[M // 2] = -1
    lp, en = ops.unembed_logprob(hid.to(DEV), emb.to(DEV), tgt.to(DEV), want_logprob=True, want_entropy=True)
    logits = bf(hid.double() @ emb.double().t())
    rlp, ren = R.op_logprob_entropy(logits, tgt)
    ulp = float(logits.abs().max()) * 2 ** -7
    assert lp[M // 2].item() == 0.0
    assert (lp.double().cpu() - rlp).abs().max() <= 2.5 * ulp and (lp.double().cpu() - rlp).abs().mean() <= 0.25 * ulp
    assert (en.double().cpu() - ren).abs().max() <= 2.5 * ulp
    only, none = ops.unembed_logprob(hid.to(DEV), emb.to(DEV), None, want_logprob=False, want_entropy=True)
    assert only is None and torch.equal(none, en)


@pytest.mark.parametrize("M,K,two", [(4095, 448, True), (4096, 448, False), (4096, 512, True), (98303, 512, True), (98304, 512, False), (98304, 768, True)])
def test_tail_on_both_sides_of_its_rule(ops, M, K, two):
    """The two forms round the same logits once: equal but where an fp32 sum in the other order crosses a rounding boundary (one bf16 step of a logit)."""
    assert ops._tail_in_two(M, K) == two
    hid, emb = bf(torch.randn(M, K, generator=gen(46))).to(DEV), bf(torch.randn(512, K, generator=gen(47)) * (4.0 / math.sqrt(K))).to(DEV)
    tgt = torch.randint(0, 512, (M,), generator=gen(48)).to(DEV)
    lp, en = ops.unembed_logprob(hid, emb, tgt, want_entropy=True)
    ops._tail_in_two = lambda M, K: not two
    try:
        lp2, en2 = ops.unembed_logprob(hid, emb, tgt, want_entropy=True)
    finally:
        del ops._tail_in_two
    ulp = 32 * 2.0 ** -7                                         # (logits of up to 5 sigma = 20)
    assert (lp - lp2).abs().max() <= 2.5 * ulp and (lp - lp2).abs().mean() <= 0.02 * ulp and (en - en2).abs().max() <= 2.5 * ulp


def test_tail_in_chunks_is_bitwise_the_whole(ops):
    hid, emb = bf(torch.randn(5000, 512, generator=gen(43))).to(DEV), bf(torch.randn(512, 512, generator=gen(44)) * 0.2).to(DEV)
    tgt = torch.randint(0, 512, (5000,), generator=gen(45)).to(DEV)
    whole = ops.unembed_logprob(hid, emb, tgt, want_entropy=True)
    ops.TAIL_ROWS = 1024
    try:
        parts = ops.unembed_logprob(hid, emb, tgt, want_entropy=True)
    finally:
        del ops.TAIL_ROWS
    assert torch.equal(whole[0], parts[0]) and torch.equal(whole[1], parts[1])


@pytest.mark.parametrize("B,T", [(1, 1), (1, 3), (1, 5), (2, 17), (1, 33), (3, 100), (1, 161), (2, 255)])
def test_hyena_on_short_segments(ops, B, T):
    """The segment chosen for the input: as near to the oracle as one segment for the whole input (state: fp32 inside and at the boundaries)."""
    D, H = 256, 2
    prm = hyena_params(D, 50)
    z = bf(torch.randn(B, T, 3 * D, generator=gen(51)))
    ry, rst = R.op_hyena(z, *prm, H)
    y, st = run_hyena(ops, z, prm, H, want_state=True)
    assert_close_bf16(y, ry)
    assert (st.cpu().to(torch.complex128) - rst).abs().max() <= 2e-5 * rst.abs().max()
