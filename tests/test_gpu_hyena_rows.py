"""GPU: which Hyena layers go channel-major (StripedHyena._hyena_ct_ok), and that both ways give the same logits and end states: two bf16 evaluations of one model
(test_gpu_packed_prompts.py: its tolerance)."""
import pytest
import torch

from oracle import stripedhyena_ref as R
from test_gpu_model import DEV, SMALL4, build, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,channels", [(1, 256, False), (8, 32, False), (3, 341, False), (1, 1023, False), (31, 33, False), (1, 513, True), (1, 1024, True), (32, 32, True), (2, 520, True)])
def test_rows(B, T, channels):
    _, _, m = build(dict(SMALL4))
    g = torch.Generator().manual_seed(B * T)
    ids = torch.tensor(list(b"ACGT"))[torch.randint(0, 4, (B, T), generator=g)].to(DEV)
    assert m._hyena_ct_ok(torch.empty(1, device=DEV), m.blocks[0], B, T) == channels
    out = []
    with torch.inference_mode():
        for other in (False, True):
            if other:
                m._hyena_ct_ok = lambda x, blk, b, t: not channels and m.ops.zt_shape_ok(b, t, *blk.projections.weight.shape)
            c = m.initialize_inference_params()
            c["mha"].max_batch_size, c["mha"].max_seqlen = B, T
            lg = m(ids, c)[0].float()
            out.append((m(ids)[0].float(), lg, *(torch.view_as_real(c["hyena"].state_dict[i]) for i in m.hyena_layer_idxs), *(c["hyena"].fir_state_dict[i].float() for i in m.hyena_layer_idxs)))
    for a, b in zip(*out):
        assert ((a - b).norm() / b.norm()).item() < 3e-2


@pytest.mark.parametrize("B,T", [(1, 256), (3, 341), (1, 513), (1, 1023), (2, 520)])
def test_both_ways_against_64_bits(B, T):
    """Logits, end states and last rows of z of either way, against the fp64 oracle: no further off than half as much again as bf16 itself (the bf16 oracle; test_gpu_model.py
    has the bound), and the token-major way no further than the channel-major one by more than that half."""
    cfg, sd, m = build(dict(SMALL4))
    g = torch.Generator().manual_seed(T)
    ids = torch.tensor(list(b"ACGT"))[torch.randint(0, 4, (B, T), generator=g)]

    def outputs(model, x, cut=lambda t: t.double().cpu()):
        c = model.initialize_inference_params()
        c["mha"].max_batch_size, c["mha"].max_seqlen = B, T
        lg = model(x, c)[0]
        h = c["hyena"]
        return [cut(lg)] + [cut(torch.view_as_real(h.state_dict[i].resolve_conj())) for i in m.hyena_layer_idxs] + [cut(h.fir_state_dict[i]) for i in m.hyena_layer_idxs]
    want = outputs(R.RefStripedHyena(cfg, sd, "fp64"), ids)
    floor = [rel_l2(a, b) for a, b in zip(outputs(R.RefStripedHyena(cfg, sd, "bf16"), ids), want)]
    err = []
    with torch.inference_mode():
        for channels in (False, True):
            m._hyena_ct_ok = lambda x, blk, b, t: channels and m.ops.zt_shape_ok(b, t, *blk.projections.weight.shape)
            err.append([rel_l2(a, b) for a, b in zip(outputs(m, ids.to(DEV)), want)])
    for f, rows, channel in zip(floor, *err):
        assert max(rows, channel) < max(1.5 * f, 4e-3), (floor, err)
        assert rows < 1.5 * channel + 1e-4, (floor, err)
