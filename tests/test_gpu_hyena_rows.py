"""GPU: which Hyena layers go channel-major (StripedHyena._hyena_ct_ok), and that both ways give the same logits and end states: two bf16 evaluations of one model
(test_gpu_packed_prompts.py: its tolerance)."""
import pytest
import torch

from test_gpu_model import DEV, SMALL4, build

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
