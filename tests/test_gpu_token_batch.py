"""The description of a batch of prompts from kernel arguments (csrc/elementwise.hip evo_token_batch), against the one made from a copy."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,past", [([1], [0]), ([300], [7]), ([255, 1, 256], [0, 0, 0]), ([0, 5, 0, 0, 700, 0], [3, 0, 0, 9, 1 << 40, 0]), ([0], [0]), ([3] * 64, list(range(64))),
                                       ([1000 - 15 * i for i in range(64)], [0] * 64), ([4] * 65, [1] * 65)])
def test_batch_of_prompts(lens, past):
    from evo_amd.mixer_ops import TokenBatch
    from evo_amd.ops import default_ops
    got, want = TokenBatch.of_prompts(lens, past, "cuda", default_ops()), TokenBatch.of_prompts(lens, past, "cpu")
    for name in ("cu", "seq", "pos", "resume"):
        a, b = getattr(got, name), getattr(want, name)
        assert (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and a.is_contiguous() and torch.equal(a.cpu(), b))), name
    assert (got.lens, got.past, got.decode) == (want.lens, want.past, want.decode)


def test_rows_of_the_host():
    from evo_amd.ops import default_ops
    for n in (0, 1, 64, 65):
        rows = [7 * i - 3 for i in range(n)]
        got = default_ops().host_rows(rows, "cuda")
        assert got.dtype == torch.int64 and got.tolist() == rows
    with pytest.raises(RuntimeError):
        default_ops().token_batch([1], [-1], "cuda")


def test_ids_that_are_not_there():
    """Looked at behind the launches of a prompt's layers: the same error, from the same call, and the next call is as if nothing had been."""
    from evo_amd.pool import DecodePool
    from evo_amd.sh.model import StripedHyena
    from evo_amd.tokenizer import CharLevelTokenizer
    model = StripedHyena(dict(vocab_size=512, hidden_size=512, num_layers=2, attn_layer_idxs=[1], num_attention_heads=4))
    g = torch.Generator().manual_seed(0)
    with torch.no_grad():
        for name, p in model.named_parameters():
            p.copy_(torch.rand(p.shape, generator=g) * 0.5 if name.endswith(("poles", "residues")) else torch.randn(p.shape, generator=g) * 0.05)
    model.to_bfloat16_except_poles_residues()
    model = model.to("cuda").eval()
    prompts = [torch.randint(0, 512, (n,), generator=g).cuda() for n in (40, 33)]
    pool = DecodePool(model, CharLevelTokenizer(512), n_slots=2)
    want = pool.prefill(prompts)
    for bad in (512, -1):
        wrong = [prompts[0], torch.cat([prompts[1][:-1], torch.tensor([bad], device="cuda")])]
        with pytest.raises(IndexError, match="outside"):
            pool.prefill(wrong)
        with pytest.raises(IndexError, match="outside"):
            pool.prefill(wrong[1:])
    for (a, _, _), (b, _, _) in zip(pool.prefill(prompts), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_ids_that_are_not_there_in_a_layered_decoder(dtype):
    """The same of LayeredDecoder's prompts, packed in one pass or several."""
    import vozalorn_util as U
    from evo_amd.ops import default_ops
    cfg = U.CONFIGS["window_64"]
    model = U.build(cfg, U.weights(cfg), dtype=dtype, device="cuda", ops=default_ops())
    g = torch.Generator().manual_seed(0)
    prompts = [torch.randint(0, cfg["vocab"], (n,), generator=g).cuda() for n in (40, 33, 70)]
    for rows in (1 << 20, 64):
        model.max_rows_per_pass = rows
        with torch.inference_mode():
            want = model.prefill_rows(prompts)
            for at in range(3):
                for bad in (cfg["vocab"], -1):
                    wrong = [p.clone() for p in prompts]
                    wrong[at][-1] = bad
                    with pytest.raises(IndexError, match="outside"):
                        model.prefill_rows(wrong)
            for (a, _, _), (b, _, _) in zip(model.prefill_rows(prompts), want):
                assert torch.equal(a, b)
