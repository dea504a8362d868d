"""CPU: ids of prompts that are looked at behind the launches of their passes (prefill_rows of either model), on embeddings whose flag is a host tensor and an event that
notes when it was waited for."""
import pytest
import torch

import vozalorn_util as U
from golden_common import TINY, tiny_model
from mixer_oracle_ops import MixerOracleOps
from oracle_ops import OracleOps

from evo_amd.ops import HipOps
from evo_amd.sh.model import StripedHyena


class Late:
    """Mixed into an op set: embeddings as launches that replace ids outside the table and raise a flag."""
    check_ids = staticmethod(HipOps.check_ids)

    def __init__(self, *args):
        super().__init__(*args)
        self.embedded, self.waited = 0, []

    def look(self, ids, vocab, later):
        bad, n = (ids < 0) | (ids >= vocab), self.embedded
        self.embedded += 1
        done = type("Event", (), {"synchronize": lambda _: self.waited.append((n, self.embedded))})()
        later.append((bad.any().to(torch.int32).reshape(1), done, vocab))
        return torch.where(bad, torch.zeros_like(ids), ids)


class Ops(Late, OracleOps):
    def embed(self, ids, weight, validate=True, later=None):
        return super().embed(self.look(ids, weight.shape[0], later), weight)


class MixerOps(Late, MixerOracleOps):
    def embed_stream(self, ids, weight, scale, validate=True, later=None):
        return super().embed_stream(self.look(ids, weight.shape[0], later), weight, scale)


def hyena():
    m = StripedHyena(dict(TINY), ops=Ops(torch.float64))
    m.load_state_dict(tiny_model().state_dict())
    return m, 512


def decoder():
    cfg = U.CONFIGS["plain"]
    m = U.build(cfg, U.weights(cfg), ops=MixerOps())
    m.max_rows_per_pass = 1                                          # a prompt a pass
    return m, cfg["vocab"]


@pytest.mark.parametrize("make", [hyena, decoder])
@pytest.mark.parametrize("at", [0, 2, 5])
@pytest.mark.parametrize("below", [False, True])
def test_one_pass_in_flight(make, at, below):
    """A pass with ids that are not there is the last but one that is launched, whatever is still to come, and the error is the call's own."""
    m, vocab = make()
    prompts = [torch.tensor([1 + i, 2, 3]) for i in range(6)]
    good = m.prefill_rows(prompts)
    assert m.ops.embedded == 6 and m.ops.waited == [(n, min(n + 2, 6)) for n in range(6)]
    wrong = [p.clone() for p in prompts]
    wrong[at][1] = -1 if below else vocab
    m.ops.embedded, m.ops.waited = 0, []
    with pytest.raises(IndexError, match=f"outside \\[0, {vocab}\\)"):
        m.prefill_rows(wrong)
    assert m.ops.embedded == min(at + 2, 6)
    for (a, _, _), (b, _, _) in zip(m.prefill_rows(prompts), good):
        assert torch.equal(a, b)
