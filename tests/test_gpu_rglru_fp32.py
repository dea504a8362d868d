"""Gated linear recurrence in fp32: the gate kernel on the matrix cores at the edges of its tiles and rules, the plain one behind them, and the scan's blocks of
eight tokens, against the reference of test_gpu_rglru.py."""
import pytest
import torch

from test_gpu_rglru import DEV, F32, decay_of, layer, ops, plain, prompt_case, rel_err, rnd, run_kernel  # noqa: F401  (ops: the fixture)

pytestmark = pytest.mark.gpu


# blocks of 256, of 20 (a step of 16 inputs and a rest of 4), 516 (three tiles of 256 channels), 1,024 and 1,028 (the last width on the matrix cores, the first off
# them); 64 tiles of 16 tokens x 4 blocks: four channel tiles a wave; 9 and 17 tokens: a block of eight in the scan and one more
@pytest.mark.parametrize("W,nb,taps", [(1024, 4, 4), (80, 4, 4), (1032, 2, 3), (1024, 1, 2), (1028, 1, 4)])
@pytest.mark.parametrize("lens", [[16], [9, 17, 39], [1, 8, 1100]])
def test_prompts(ops, W, nb, taps, lens):
    prompt_case(ops, F32, lens, W, nb, taps, past=[3] * len(lens), seed=11)


@pytest.mark.parametrize("B", [3, 64, 65])
@pytest.mark.parametrize("W,nb", [(1024, 4), (1032, 2), (12, 3)])
def test_one_step(ops, W, nb, B):
    from evo_amd.mixer_ops import TokenBatch
    w, taps = layer(W, nb, 2, F32, 5), 2
    state, z = rnd(B, 1 + taps, W, seed=8), rnd(B, 2 * W, seed=9)
    st = state.to(DEV)
    o = run_kernel(ops, z, None, False, W, w, TokenBatch.of_decode(torch.full((B,), 4, device=DEV)), st)
    for b in (0, B - 1):
        want, _, last = plain(z[b:b + 1, W:].double(), z[b:b + 1, :W].double(), w, state[b, 1 + 3 % taps][None].double(), state[b, 0].double())
        assert rel_err(o[b:b + 1], want) < 5e-6 and rel_err(st[b:b + 1, 0], last[None]) < 5e-6
