"""GPU: StripedHyena prompts of fewer than 32 tokens in a pool keep the modal kernels (fp32 states; the matrix-core operator holds filters and states as bf16 hi + lo): the
bits of the same prompt alone, whoever is admitted beside it."""
import pytest
import torch

from test_gpu_model import SMALL4, build
from test_gpu_packed_prompts import WIDE, prompts_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,lens", [("toy", [4, 5, 31]), ("toy", [100, 3, 8, 40, 31, 1, 65]), ("wide", [31, 16, 8, 64, 64])])
def test_short_prompts(dims, lens):
    _, _, m = build(dict(SMALL4 if dims == "toy" else WIDE))
    prompts = prompts_of(lens)
    with torch.inference_mode():
        together = m.prefill_rows(prompts)
        for n, p, (lg, ipd, row) in zip(lens, prompts, together):
            if n >= 32:
                continue
            alone_lg, alone, r = m.prefill_rows([p])[0]
            assert torch.equal(lg, alone_lg), n
            assert torch.equal(ipd["mha"].key_value_memory_dict[1][row, :n], alone["mha"].key_value_memory_dict[1][r, :n])
            for i in m.hyena_layer_idxs:
                for a, b in ((ipd["hyena"].state_dict, alone["hyena"].state_dict), (ipd["hyena"].fir_state_dict, alone["hyena"].fir_state_dict)):
                    a, b = (t[k] for t, k in ((a[i], row), (b[i], r)))
                    assert torch.equal(torch.view_as_real(a) if a.is_complex() else a, torch.view_as_real(b) if b.is_complex() else b), (n, i)
