"""A norm between two weight-streaming layers without a launch of its own (csrc/gemv.hip skinny_kw_kernel EP 3, skinny_ring_kernel RS)."""
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
    return (torch.randn(*shape, generator=g) * scale).to(DEV, BF)


@pytest.mark.parametrize("M,N,K", [(5, 2048, 1152), (8, 4096, 11008), (9, 4096, 4096), (16, 3072, 8320), (17, 4096, 4096), (32, 2112, 7040)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_layer_residual_and_scaled_rows(ops, M, N, K, with_bias):
    """The new rows are linear_residual_'s bits; their scaled copy and sums of squares follow from them (16 squares: 2^-20 of their sum)."""
    a, w, x, scale = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(M, N, seed=3), rnd(N, seed=4)
    bias = rnd(N, seed=5) if with_bias else None
    want = ops.linear_residual_(x.clone(), a, w, bias=bias)
    xg, ss = ops.linear_residual_scaled_(x, a, w, bias, scale)
    assert torch.equal(x, want) and torch.equal(xg, (want.float() * scale.float()).to(BF))
    sums = want.double().square().view(M, N // 16, 16).sum(-1)
    assert ((ss.double() - sums).abs() <= 2.0 ** -20 * sums).all()


def norm64(x, scale, eps):
    return x.double() / (x.double().square().mean(-1, keepdim=True).sqrt() + eps) * scale.double()


def bound(x, xg, f, w):
    """Of the product of bf16(x scale): half an ulp of each of its values, 2^-9, and K 2^-24 for fp32 sums."""
    K = w.shape[1]
    return (xg.double().abs() * f) @ w.double().abs().T * (2.0 ** -9 + K * 2.0 ** -24)


@pytest.mark.parametrize("M", [5, 8, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(4160, 2048), (6144, 4096), (8192, 2176), (12288, 4096), (16384, 3072), (24576, 4096)])
def test_layer_on_row_factors(ops, M, N, K):
    x, scale, w, b = rnd(M, K, seed=1, scale=3.0), rnd(K, seed=2), rnd(N, K, seed=3, scale=K ** -0.5), rnd(N, seed=4)
    if not ops.factors_ok(M, w):                                 # (layers in parts of K: 17 rows and more of up to 8,192 columns)
        assert M > 16 and ops.lib.evo_linear_parts(M, N, K) > 0
        return
    x[0] = 0                                                     # eps alone
    xg, ss = (x.float() * scale.float()).to(BF), x.float().square().view(M, K // 16, 16).sum(-1).contiguous()
    f = 1.0 / (x.double().square().mean(-1, keepdim=True).sqrt() + 1e-6)
    for bias in (None, b):
        got = ops.linear_factors(xg, ss, 1e-6, w, bias).double()
        want = norm64(x, scale, 1e-6) @ w.double().T + (0 if bias is None else bias.double())
        assert ((got - want).abs() <= bound(x, xg, f, w) + want.abs() * 2.0 ** -8).all()


@pytest.mark.parametrize("M", [5, 16, 32])
@pytest.mark.parametrize("I,K", [(2112, 2048), (4096, 4096), (5504, 2048), (11008, 4096)])
def test_gate_on_row_factors(ops, M, I, K):
    x, scale, w12 = rnd(M, K, seed=1, scale=3.0), rnd(K, seed=2), rnd(2 * I, K, seed=3, scale=K ** -0.5)
    xg, ss = (x.float() * scale.float()).to(BF), x.float().square().view(M, K // 16, 16).sum(-1).contiguous()
    f = 1.0 / (x.double().square().mean(-1, keepdim=True).sqrt() + 1e-6)
    assert ops.factors_ok(M, w12, gate=True)
    z = norm64(x, scale, 1e-6) @ w12.double().T
    z1, z2 = z[:, :I], z[:, I:]
    want, err = torch.nn.functional.gelu(z1) * z2, bound(x, xg, f, w12) + z.abs() * 2.0 ** -9      # (both halves rounded; the gate's slope is at most 1.13)
    e1, e2 = 1.13 * err[:, :I], err[:, I:]
    limit = e1 * z2.abs() + torch.nn.functional.gelu(z1).abs() * e2 + e1 * e2 + want.abs() * 2.0 ** -7 + 1e-3
    plain = ops.mlp_gate_factors(xg, ss, 1e-6, w12, False)
    assert ((plain.double() - want).abs() <= limit).all()
    assert torch.equal(ops.mlp_gate_factors(xg, ss, 1e-6, ops.pack_gate_weights(w12), True), plain)


def test_what_stays(ops):
    def takes(M, N, K):
        return ops.linear_residual_scaled_(rnd(M, N, seed=1), rnd(M, K, seed=2), rnd(N, K, seed=3), None, rnd(N, seed=4)) is not None
    assert takes(16, 4096, 4096)
    for shape in ((4, 4096, 4096), (33, 4096, 4096), (17, 4096, 8192), (16, 4160, 4096), (16, 2080, 4096), (16, 1984, 4096), (16, 4096, 1024), (16, 4096, 4128)):
        assert not takes(*shape)
    for M, N, K in ((4, 12288, 4096), (33, 12288, 4096), (16, 4096, 4096), (16, 24640, 4096), (16, 12288, 4224), (16, 12288, 1920)):
        assert not ops.factors_ok(M, rnd(N, K, seed=1))


@pytest.mark.parametrize("B", [5, 16, 20])
def test_decode_steps_of_a_pool(ops, B, monkeypatch):
    """Steps whose layers hand the next norm on, against the same with every norm in its own launch: a norm's rows are rounded before their factor, not behind it."""
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
    ids = torch.randint(0, 512, (B, 12), generator=g).to(DEV)
    calls = []
    was = type(ops).linear_residual_scaled_

    def steps():
        ipd = model.initialize_inference_params()
        ipd["mha"].max_batch_size = ipd["hyena"].max_batch_size = B
        out = [model(ids[:, :8], inference_params_dict=ipd)[0][:, -1:]]
        for t in range(8, 12):
            ipd["mha"].seqlen_offset = ipd["hyena"].seqlen_offset = t
            out.append(model(ids[:, t:t + 1], inference_params_dict=ipd)[0])
        return torch.cat(out, 1).float()
    with torch.inference_mode():
        monkeypatch.setattr(type(ops), "linear_residual_scaled_", lambda self, *a: calls.append(was(self, *a)) or calls[-1])
        got = steps()
        assert sum(c is not None for c in calls) >= 3
        monkeypatch.setattr(type(ops), "linear_residual_scaled_", lambda *a: None)
        model._dgraph = None
        want = steps()
    assert ((got - want).norm() / want.norm()).item() < 12 * 2.0 ** -9     # (six norms a step, each rounded once, 2^-9 at most, on either side)


@pytest.mark.parametrize("B,width", [(40, 2048), (24, 4096)])
def test_decode_steps_that_add_parts(ops, B, width, monkeypatch):
    """Steps of 17 to 64 rows, whose norms add the parts of the layers in front of them (at 24 rows of 4,096 the mixer's, as row factors, in between): the same bits eagerly and
    captured, and every norm's rows against its own launch's."""
    from evo_amd.sh.model import StripedHyena
    model = StripedHyena(dict(vocab_size=512, hidden_size=width, num_layers=3, attn_layer_idxs=[1], num_attention_heads=width // 128))
    g = torch.Generator(device=DEV).manual_seed(0)
    model.to_bfloat16_except_poles_residues()
    model = model.to(DEV).eval()
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith(("poles", "residues")):
                p.uniform_(0.0, 0.5, generator=g)
            else:
                p.normal_(1.0 if name.endswith("scale") else 0.0, 0.02 if p.dim() > 1 else 0.1, generator=g)
    ids = torch.randint(0, 512, (B, 13), generator=g, device=DEV)
    added, scaled, one = [], [], []
    norm_, scaled_ = type(ops).linear_residual_norm_, type(ops).linear_residual_scaled_

    def steps(captured):
        model.decode_graph, model._dgraph, model._dgraph_warm, model.decode_graph_replays = captured, None, None, 0
        ipd = model.initialize_inference_params()
        ipd["mha"].max_batch_size = ipd["hyena"].max_batch_size = B
        ipd["mha"].max_seqlen = 16
        out = [model(ids[:, :8], inference_params_dict=ipd)[0][:, -1:]]
        for t in range(8, 13):
            one.append(1)
            ipd["mha"].seqlen_offset = ipd["hyena"].seqlen_offset = t
            out.append(model(ids[:, t:t + 1], inference_params_dict=ipd)[0])
            if captured:                                             # (eager work between the replays)
                ops.rmsnorm(out[-1].new_ones(3, 512), None, out[-1].new_ones(512), 1e-6)
                torch.cuda.synchronize()
            one.pop()
        assert not captured or model.decode_graph_replays >= 3
        return torch.cat(out, 1).float()
    with torch.inference_mode():
        monkeypatch.setattr(type(ops), "linear_residual_norm_", lambda self, *a, **k: ((got := norm_(self, *a, **k)), added.append(got) if one and got is not None else None)[0])
        monkeypatch.setattr(type(ops), "linear_residual_scaled_", lambda self, *a: ((got := scaled_(self, *a)), scaled.append(got) if one and got is not None else None)[0])
        got = steps(False)
        assert len(added) >= 5 * 3 and (len(scaled) >= 5 * 3) == (B <= 32)      # (a step: three layers' at least)
        assert torch.equal(steps(True), got)
        monkeypatch.setattr(type(ops), "linear_residual_norm_", lambda *a, **k: None)
        monkeypatch.setattr(type(ops), "linear_residual_scaled_", lambda *a: None)
        want = steps(False)
    assert ((got - want).norm() / want.norm()).item() < 12 * 2.0 ** -9     # (as above)
