"""Launches that took over what stood behind them in a decode step: closing norms on the parts of a dense layer, decode attention that writes its own result."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from evo_amd.ops import default_ops
    return default_ops()


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale)


@pytest.mark.parametrize("M,N,K", [(17, 4096, 8192), (24, 1024, 11008), (32, 4096, 16384), (33, 4096, 4096), (64, 1088, 1024), (64, 3072, 8320)])
@pytest.mark.parametrize("alpha", [None, 2.0])
def test_closing_norm_of_parts(ops, M, N, K, alpha):
    """The same bits as the layer with its sum rounded by itself and the closing norm behind it; a norm weight at an odd place takes those."""
    a, w = rnd(M, K, seed=1).to(DEV, BF), rnd(N, K, seed=2, scale=K ** -0.5).to(DEV, BF)
    for g in (rnd(N, seed=3).to(DEV, BF), rnd(N + 1, seed=4).to(DEV, BF)[1:]):
        x, xb = rnd(M, N, seed=5).to(DEV), torch.zeros(M, N, device=DEV, dtype=BF)
        x2, xb2 = x.clone(), xb.clone()
        parts = ops.linear_parts(a, w)
        assert parts is not None and parts.dim() == 3
        ops.closing_parts_(x, xb, parts, g, alpha, 1e-6, 1.0)
        y = ops.linear(a, w)
        if alpha is None:
            ops.postnorm_residual_(x2, xb2, y, g, 1e-6, 1.0)
        else:
            ops.sum_norm_(x2, xb2, y, g, alpha, 1e-6, 1.0)
        assert torch.equal(x, x2) and torch.equal(xb, xb2)


@pytest.mark.parametrize("M,D,dtype", [(1, 2048, BF), (3, 4096, torch.float32), (5, 4096, BF), (2, 8192, torch.float32), (300, 8192, BF)])
@pytest.mark.parametrize("alpha", [None, 2.0])
def test_last_closing_norm_with_the_final_one(ops, M, D, dtype, alpha):
    """The same bits as the closing norm and the final norm in launches of their own; the stream stays as it was."""
    x, y, g, wf = (rnd(*s, seed=i).to(DEV, t) for i, (s, t) in enumerate((((M, D), torch.float32), ((M, D), dtype), ((D,), dtype), ((D,), dtype))))
    was = x.clone()
    assert ops.closing_final_ok(y, g, x, wf)
    got = ops.closing_final(x, y, g, wf, alpha, 1e-6, 1.0)
    assert torch.equal(x, was)
    xb = x if dtype == torch.float32 else torch.zeros(M, D, device=DEV, dtype=BF)
    if alpha is None:
        ops.postnorm_residual_(x, xb, y, g, 1e-6, 1.0)
    else:
        ops.sum_norm_(x, xb, y, g, alpha, 1e-6, 1.0)
    assert torch.equal(got, ops.rmsnorm_stream(x, wf, 1e-6, 1.0))
    assert not ops.closing_final_ok(y[:, 8:].contiguous(), g[8:], x[:, 8:].contiguous(), wf[8:])
    parts = rnd(7, M, 4096, seed=9).to(DEV)
    x, xb, g, wf = (t[..., :4096].contiguous() if t.shape[-1] > 4096 else torch.nn.functional.pad(t, (0, 4096 - t.shape[-1])) for t in (was, xb.to(BF), g.to(BF), wf.to(BF)))
    for n in (1, 2, 3, 4, 7):
        x2, xb2 = x.clone(), torch.zeros_like(xb)
        got = ops.closing_final(x, parts[:n], g, wf, alpha, 1e-6, 1.0)
        ops.closing_parts_(x2, xb2, parts[:n], g, alpha, 1e-6, 1.0)
        assert torch.equal(got, ops.rmsnorm_stream(x2, wf, 1e-6, 1.0))


@pytest.mark.parametrize("D", [2048, 4096, 8192])
@pytest.mark.parametrize("dtype", [BF, torch.float32])
def test_rows_of_whole_runs(ops, D, dtype):
    """Rows that a thread requests whole against rows that it walks: D elements and 15 D zeros behind them, a row no form has whole runs of.  A thread has the same elements in the same
    order and then zeros, so the sum of squares is the same number; its mean over 16 D and a sixteenth of eps make a root of a quarter and four times the norm, all exactly.  Only where
    that is added to the stream does either side round once more: 2^-24 of its result."""
    M = 5
    x, y, g = (rnd(*s, seed=i).to(DEV, t) for i, (s, t) in enumerate((((M, D), torch.float32), ((M, D), dtype), ((D,), dtype))))

    def wide(t):
        return torch.nn.functional.pad(t, (0, 15 * D))
    for alpha in (None, 2.0):
        a, b = x.clone(), wide(x)
        ab, bb = (a, b) if dtype == torch.float32 else (torch.zeros_like(y), torch.zeros_like(wide(y)))
        if alpha is None:
            ops.postnorm_residual_(a, ab, y, g, 1e-6, 1.0)
            ops.postnorm_residual_(b, bb, wide(y), wide(g), 1e-6 / 16, 1.0)
            b = b[:, :D].double()
            assert ((a.double() - (x.double() + (b - x.double()) / 4)).abs() <= 2.0 ** -24 * (a.double().abs() + b.abs() / 4)).all()
        else:
            ops.sum_norm_(a, ab, y, g, alpha, 1e-6, 1.0)
            ops.sum_norm_(b, bb, wide(y), wide(g), alpha, 1e-6 / 16, 1.0)
            assert torch.equal(4 * a, b[:, :D])
        assert torch.equal(ab, a.to(dtype))
    assert torch.equal(4 * ops.rmsnorm_stream(x, g, 1e-6, 1.0), ops.rmsnorm_stream(wide(x), wide(g), 1e-6 / 16, 1.0)[:, :D])
    z = rnd(M, D, seed=7).to(DEV, dtype)
    assert torch.equal(4 * ops.gated_norm(y, z, g, 1e-6), ops.gated_norm(wide(y), wide(z), wide(g), 1e-6 / 16)[:, :D])


@pytest.mark.parametrize("D,counts", [(2048, (513, 4096, 4097)), (4096, (513, 4097)), (8192, (256, 257, 401, 900, 901, 513, 1024, 1025))])
@pytest.mark.parametrize("dtype", [BF, torch.float32])
def test_rows_of_either_form(ops, D, counts, dtype):
    """Rows of a count that takes the loop, or the row at once, against the same rows 200 at a time: a thread has the same elements in the same order, so the same bits."""
    for M in counts:
        x, y, z, g = (rnd(*s, seed=i).to(DEV, t) for i, (s, t) in enumerate((((M, D), torch.float32), ((M, D), dtype), ((M, D), dtype), ((D,), dtype))))
        for norm in (lambda x, xb, y: ops.sum_norm_(x, xb, y, g, 2.0, 1e-6, 1.0), lambda x, xb, y: ops.postnorm_residual_(x, xb, y, g, 1e-6, 1.0)):
            a, b = x.clone(), x.clone()
            ab, bb = (a, b) if dtype == torch.float32 else (torch.zeros_like(y), torch.zeros_like(y))
            norm(a, ab, y)
            for at in range(0, M, 200):
                bp = b[at:at + 200]
                norm(bp, bp if bb is b else bb[at:at + 200], y[at:at + 200])
            assert torch.equal(a, b) and torch.equal(ab, bb)
        assert torch.equal(ops.gated_norm(y, z, g, 1e-6), torch.cat([ops.gated_norm(y[at:at + 200], z[at:at + 200], g, 1e-6) for at in range(0, M, 200)]))


def test_one_sum_stays_one_sum(ops):
    for M, N, K in ((16, 4096, 16384), (24, 4096, 4096), (65, 4096, 16384), (24, 4160, 16384), (24, 4096, 16416), (24, 512, 16384)):
        assert ops.linear_parts(torch.zeros(M, K, device=DEV, dtype=BF), torch.zeros(N, K, device=DEV, dtype=BF)) is None
    assert ops.linear_parts(torch.zeros(24, 8192, device=DEV), torch.zeros(4096, 8192, device=DEV)) is None


@pytest.mark.parametrize("H,G,maps,n,dv,ring", [(4, 4, 1, 128, 128, 40), (6, 2, 1, 56, 40, 129), (16, 1, 1, 64, 64, 300), (40, 2, 1, 64, 128, 64), (2, 1, 1, 256, 256, 33),
                                                (8, 1, 2, 64, 64, 200), (3, 3, 2, 56, 112, 500), (2, 2, 2, 128, 256, 130)])
def test_decode_attention_in_one_launch(ops, H, G, maps, n, dv, ring, monkeypatch):
    """Against one part and its merge: the same sums, divided and combined in another order, rounded once (bf16: half an ulp is 2^-9 of the value, two roundings of
    nearly the same number differ by at most one ulp, 2^-7 of the smaller one)."""
    B = 5
    z = rnd(B, (H + G) * maps * n + G * dv, seed=1, scale=2.0).to(DEV, BF)
    z = torch.nn.functional.pad(z, (0, -z.shape[1] % 8))
    cache = rnd(B, ring, (G * (maps * n + dv) + 7) // 8 * 8, seed=2).to(DEV, BF)
    pos = torch.tensor([0, 31, 32, ring - 1, 3 * ring], device=DEV)
    args = (z, cache, pos, H, G, maps, n, dv, n ** -0.5, 0.45, 0.7, 1e-4)
    want = ops.heads_decode(*args, n_split=1).float()
    whole = ops.heads_whole_ok
    assert whole(160, ring, H // G, maps, n, dv, z, cache) and not whole(79, ring, H // G, maps, n, dv, z, cache)
    names = []
    real = ops._t
    monkeypatch.setattr(ops, "heads_whole_ok", lambda *a: True, raising=False)
    monkeypatch.setattr(ops, "_t", lambda name: (names.append(name), real(name))[1], raising=False)
    got = ops.heads_decode(*args).float()
    assert names == ["heads_decode_whole"]
    assert bool(((got - want).abs() <= want.abs() * 2.0 ** -7 + 1e-5).all()), (got - want).abs().max().item()
    assert (got != want).float().mean() < 0.02


def test_what_one_launch_refuses(ops):
    z, cache, pos = torch.zeros(2, 17 * 2 * 64, device=DEV, dtype=BF), torch.zeros(2, 16, 192, device=DEV, dtype=BF), torch.zeros(2, dtype=torch.int64, device=DEV)
    o = torch.zeros(2, 17 * 64, device=DEV, dtype=BF)
    assert not ops.heads_whole_ok(1000, 16, 17, 2, 64, 64, z, cache)
    assert ops.lib.evo_heads_decode_whole(z.data_ptr(), z.stride(0), cache.data_ptr(), pos.data_ptr(), o.data_ptr(), 2, 17, 1, 2, 64, 64, 16, 192, 0.1, 0.5, 0.5, 1e-5, None) == -1


@pytest.mark.parametrize("S,V", [(1, 512), (3, 37), (300, 512), (16, 1001)])
def test_end_of_a_step(ops, S, V):
    logits = rnd(S, V, seed=1).to(DEV, BF)
    pos = torch.arange(S, device=DEV) + 95
    out = ops.step_out(logits, pos, 99)
    assert torch.equal(out, logits.float()) and torch.equal(pos.cpu(), (torch.arange(S) + 96).clamp(max=99))
    odd = logits.reshape(-1)[1:]                                  # (not 16-byte aligned)
    assert torch.equal(ops.step_out(odd, pos, 99), odd.float())


@pytest.mark.parametrize("first", [0, 1 << 30])
@pytest.mark.parametrize("B,Tq,past", [(1, 129, 0), (2, 255, 0), (1, 256, 0), (3, 257, 0), (1, 513, 0), (2, 140, 300), (1, 300, 1)])
def test_both_prompt_attention_kernels(ops, B, Tq, past, first, monkeypatch):
    """The kernel of many keys and that of few, either side of `attn_w64_from`, against fp64.  Both round the probabilities and the result to bf16: 2^-9 of it each, and
    the largest error by an outlier's share of a row (measured 2.3e-3 of the norm)."""
    monkeypatch.setattr(ops, "attn_w64_from", first, raising=False)
    H, Tk = 4, Tq + past
    q, k, v = (rnd(B, n, H, 128, seed=i, scale=s).to(DEV, BF) for i, (n, s) in enumerate(((Tq, 0.2), (Tk, 1.0), (Tk, 1.0))))
    seen = torch.arange(Tk, device=DEV)[None] <= torch.arange(Tq, device=DEV)[:, None] + past
    s = (q.double().transpose(1, 2) @ k.double().permute(0, 2, 3, 1).contiguous()) * 0.6931471805599453                    # (scores are exponents of two)
    want = (s.masked_fill(~seen, float("-inf")).softmax(-1) @ v.double().transpose(1, 2).contiguous()).transpose(1, 2)
    got = ops.attention(q, k, v, past, prescaled=True).double()
    assert (got - want).norm() / want.norm() < 4e-3
