"""CPU: programs' own versions of a model's `hidden_states` and of an op set's embeddings, with the arguments that these have always had: scorers, row groups and prompt
passes call them as they stand, whatever keywords the framework's own versions have gained."""
import functools
import types

import pytest
import torch

from golden_common import TINY, tiny_model
from oracle_ops import OracleOps

from evo_amd import scoring
from evo_amd.mixer_ops import Stream, takes
from evo_amd.sh.model import StripedHyena
from evo_amd.tokenizer import CharLevelTokenizer

PROMPTS = [[65, 67, 71], [84] * 7, [65]]


class Narrow(StripedHyena):
    """Counts its passes."""
    passes = 0

    def hidden_states(self, x, inference_params_dict=None, padding_mask=None):
        self.passes += 1
        return super().hidden_states(x, inference_params_dict, padding_mask)


class NarrowOps(OracleOps):
    """An op set with late checks of ids whose embedding does not know of them."""
    check_ids = staticmethod(lambda later: None)

    def embed(self, ids, weight):
        return OracleOps.embed(self, ids, weight)


def models():
    plain = tiny_model()
    out = []
    for cls, ops in ((Narrow, OracleOps(torch.float64)), (StripedHyena, NarrowOps(torch.float64)), (Narrow, NarrowOps(torch.float64))):
        m = cls(dict(TINY), ops=ops)
        m.load_state_dict(plain.state_dict())
        out.append(m)
    return plain, out


def test_prompt_passes():
    plain, others = models()
    want = plain.prefill_rows([torch.tensor(p) for p in PROMPTS])
    for m in others:
        for (a, _, _), (b, _, _) in zip(m.prefill_rows([torch.tensor(p) for p in PROMPTS]), want):
            assert torch.equal(a, b)
        assert not isinstance(m, Narrow) or m.passes == len(PROMPTS)


@pytest.mark.parametrize("known", [False, True])
def test_row_groups(known):
    plain, others = models()
    ids = torch.randint(0, 512, (3, 5), generator=torch.Generator().manual_seed(0))
    want = plain.hidden_states(ids, ids_known=known)
    for m in others:
        m.max_rows_per_pass = 5
        got = m.hidden_states(ids) if isinstance(m, Narrow) else m.hidden_states(ids, ids_known=known)
        assert torch.equal(got, want) and (not isinstance(m, Narrow) or m.passes == 4)


def test_scorers():
    asked = []

    class Model(types.SimpleNamespace):
        embedding_rows = 512

        def hidden_states(self, ids, inference_params_dict=None, padding_mask=None):
            asked.append(tuple(ids.shape))
            return torch.zeros(ids.numel(), 4)
    ops = types.SimpleNamespace(name="hip-gfx950", unembed_logprob_ok=lambda h, e: True,
                                unembed_logprob=lambda h, e, t, want_logprob, want_entropy: (torch.zeros(len(h)), torch.zeros(len(h)) if want_entropy else None))
    m = Model(ops=ops, hidden_size=4, unembed=types.SimpleNamespace(weight=torch.zeros(512, 4)))
    tok = CharLevelTokenizer(512)
    assert len(scoring.score_sequences(["ACGT", "AC"], m, tok, device="cpu")) == 2
    assert [len(e) for e in scoring.positional_entropies(["ACGT", "AC"], m, tok, device="cpu")] == [4, 2]
    assert asked == [(2, 5)] * 2


@pytest.mark.parametrize("known,later", [(True, None), (False, [])])
def test_residual_streams(known, later):
    class Ops:
        def embed_stream(self, ids, weight, scale):
            return weight[ids] * scale, weight[ids] * scale
    s = Stream(Ops(), torch.tensor([1, 2]), torch.eye(4), 2.0, 1e-6, 0.0, None, known, later)
    assert torch.equal(s.x, 2 * torch.eye(4)[1:3])


def test_whether_a_method_takes_a_keyword():
    def own(x, later=None): return x
    def open_(x, **more): return x
    def narrow(x): return x
    wraps_own, wraps_narrow, hides = functools.wraps(own)(lambda *a, **k: own(*a, **k)), functools.wraps(narrow)(lambda *a, **k: narrow(*a, **k)), functools.wraps(own)(lambda x: own(x))
    assert takes(own, "later") and takes(open_, "later") and takes(wraps_own, "later") and takes(torch.no_grad()(own), "later")
    assert not any(takes(f, "later") for f in (narrow, wraps_narrow, hides, functools.partial(own), len, None))
    def local(x):
        later = x
        return later
    assert not takes(local, "later")
