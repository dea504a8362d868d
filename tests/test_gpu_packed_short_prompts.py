"""GPU: StripedHyena prompts of a few tokens in a shared pass (StripedHyena._prompt_groups): who shares with whom, and the same results as alone
(test_gpu_packed_prompts.py: its comparison and its tolerance)."""
import pytest

from test_gpu_model import SMALL4, build

pytestmark = pytest.mark.gpu


def test_groups():
    _, _, m = build(dict(SMALL4))
    for lens, want in (([4, 5, 31], [[0, 1, 2]]), ([31, 8], [[0], [1]]), ([8, 32], [[0, 1]]), ([100, 3, 8, 4097, 40, 1], [[0, 2, 4], [1], [3], [5]]),
                       ([3, 2, 1], [[0], [1], [2]]), ([4096] * 17, [list(range(16)), [16]])):
        got = m._prompt_groups(lens)
        assert sorted(got) == sorted(want) and sorted(n for g in got for n in g) == list(range(len(lens)))


@pytest.mark.parametrize("dims,lens", [("toy", [4, 31, 5, 3, 8, 4097, 16]), ("wide", [4, 7, 16, 31]), ("wide", [24, 1, 100, 5])])
def test_short_prompts_together(dims, lens):
    from test_gpu_packed_prompts import test_packed_prompts_are_the_prompts_alone
    test_packed_prompts_are_the_prompts_alone(dims, lens)
