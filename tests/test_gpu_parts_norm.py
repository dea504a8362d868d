"""Dense layers in parts of K that the norm behind them adds (csrc/gemm_tile.hip evo_dense_parts_bf16, csrc/elementwise.hip evo_rmsnorm_parts_bf16)."""
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
    return torch.randn(*shape, generator=g) * scale


def in_order(parts):
    total = parts[0].clone()
    for p in parts[1:]:
        total += p
    return total


@pytest.mark.parametrize("M,D,n", [(1, 8, 1), (3, 520, 3), (2, 2048, 8), (5, 2056, 4), (17, 4096, 5), (2, 4104, 7), (161, 8192, 3), (1, 8184, 64)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_rmsnorm_adds_parts(ops, M, D, n, with_bias):
    """The bits of the sum by itself -- parts in their order, bias, residual, one rounding -- and of the norm's own launch on it."""
    part, x, scale = rnd(n, M, D, seed=1).to(DEV), rnd(M, D, seed=2).to(DEV, BF), rnd(D, seed=3).to(DEV, BF)
    bias = rnd(D, seed=4).to(DEV, BF) if with_bias else None
    total = in_order(part)
    want = ((total + bias.float() if with_bias else total) + x.float()).to(BF)
    out = torch.empty_like(x)
    from evo_amd.ops import _stream
    rc = ops.lib.evo_rmsnorm_parts_bf16(x.data_ptr(), part.data_ptr(), n, bias.data_ptr() if with_bias else None, scale.data_ptr(), out.data_ptr(), M, D, 1e-6, _stream())
    assert rc == 0 and torch.equal(x, want) and torch.equal(out, ops.rmsnorm(want, None, scale, 1e-6))


@pytest.mark.parametrize("M,N,K", [(17, 4096, 11008), (64, 4096, 16384), (65, 4096, 4096), (65, 8192, 8192), (97, 2048, 4096), (161, 4096, 11008), (192, 4096, 16384), (255, 8192, 4096),
                                   (300, 4096, 11008), (511, 2048, 5504), (700, 4096, 4096), (1023, 4096, 11008)])
def test_layer_residual_and_norm(ops, M, N, K):
    """Parts against the fp64 product (each row's fp32 sum of K products is within K 2^-24 of the sum of their magnitudes), and what is made of them against them, bit for bit."""
    a, w, bias = rnd(M, K, seed=1).to(DEV, BF), rnd(N, K, seed=2, scale=K ** -0.5).to(DEV, BF), rnd(N, seed=3).to(DEV, BF)
    scale, x = rnd(N, seed=4).to(DEV, BF), rnd(M, N, seed=5).to(DEV, BF)
    parts = ops.layer_parts(a, w)
    assert parts is not None and 2 <= parts.shape[0] <= 8
    total = in_order(parts)
    want = a.double() @ w.double().t()
    assert ((total - want).abs() <= K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t())).all()
    new = ((total + bias.float()) + x.float()).to(BF)
    got = ops.linear_residual_norm_(x, a, w, bias, scale, 1e-6)
    assert torch.equal(x, new) and torch.equal(got, ops.rmsnorm(new, None, scale, 1e-6))


def test_what_stays_in_launches_of_its_own(ops):
    def layer(M, N, K, odd=False):
        x, scale = torch.zeros(M, N, device=DEV, dtype=BF), torch.zeros(N + 1, device=DEV, dtype=BF)
        return ops.linear_residual_norm_(x, torch.zeros(M, K, device=DEV, dtype=BF), torch.zeros(N, K, device=DEV, dtype=BF), None, scale[1:] if odd else scale[:N], 1e-6)
    assert layer(161, 4096, 11008) is not None and layer(161, 4096, 11008, odd=True) is None
    for shape in ((16, 4096, 11008), (24, 4096, 4096), (1024, 4096, 11008), (161, 4160, 11008), (161, 4096, 11040), (161, 4096, 512), (161, 16384, 4096)):
        assert layer(*shape) is None


@pytest.mark.parametrize("lens", [[160], [90, 31], [299, 200]])
@pytest.mark.parametrize("cached", [False, True])
def test_scored_and_prefilled_rows(ops, lens, cached, monkeypatch):
    """A model whose layers hand the next norm on, against the same with every norm in its own launch: both within bf16's rounding of each other, layer after layer.  `cached`: a
    prompt and its continuation on states that the first call left."""
    from evo_amd.sh.model import StripedHyena
    cfg = dict(vocab_size=512, hidden_size=2048, num_layers=3, attn_layer_idxs=[1], num_attention_heads=16)
    model = StripedHyena(cfg)
    g = torch.Generator().manual_seed(0)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith(("poles", "residues")):
                p.copy_(torch.rand(p.shape, generator=g) * 0.5)
            else:
                p.copy_(torch.randn(p.shape, generator=g) * (0.02 if p.dim() > 1 else 0.1) + (1.0 if name.endswith("scale") else 0.0))
    model.to_bfloat16_except_poles_residues()
    model = model.to(DEV).eval()
    ids = torch.randint(0, 512, (len(lens), max(lens) + 1), generator=g).to(DEV)
    taken = []
    was = type(ops).linear_residual_norm_
    monkeypatch.setattr(type(ops), "linear_residual_norm_", lambda self, *a, **k: taken.append(was(self, *a, **k)) or taken[-1])

    def logits():
        if not cached:
            return model(ids)[0].float()
        ipd, half = model.initialize_inference_params(), ids.shape[1] * 3 // 5
        ipd["mha"].max_batch_size = ipd["hyena"].max_batch_size = len(lens)
        first = model(ids[:, :half], inference_params_dict=ipd)[0]
        ipd["mha"].seqlen_offset = ipd["hyena"].seqlen_offset = half
        return torch.cat([first, model(ids[:, half:], inference_params_dict=ipd)[0]], 1).float()
    with torch.inference_mode():
        got = logits()
        assert sum(t is not None for t in taken) >= (6 if cached else 3)
        monkeypatch.setattr(type(ops), "linear_residual_norm_", lambda *a, **k: None)
        want = logits()
    assert ((got - want).norm() / want.norm()).item() < 8 * 2.0 ** -9      # (six roundings of the stream, each 2^-9 of it at most)
