"""GPU: the decode pool's tokens and positions as kernel arguments (csrc/elementwise.hip), against plain indexing."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64])
def test_put_tokens(n):
    from evo_amd.ops import default_ops
    ops = default_ops()
    ids = torch.arange(1000, 1070, device="cuda")[:, None].contiguous()
    want = ids.clone()
    slots = torch.randperm(70)[:n].tolist()
    tokens = [(1 << 40) * (i % 3) - i for i in range(n)]
    ops.put_tokens(ids, slots, tokens)
    want[torch.tensor(slots).cuda(), 0] = torch.tensor(tokens).cuda()
    assert torch.equal(ids, want)


def test_put_tokens_refuses_slots_outside():
    from evo_amd.ops import default_ops
    ops = default_ops()
    ids = torch.zeros(4, 1, dtype=torch.int64, device="cuda")
    for slots in ([4], [-1], list(range(65))):
        with pytest.raises(RuntimeError):
            ops.put_tokens(ids, slots, [1] * len(slots))
    assert not ids.any()


def test_tokens_of_other_kinds():
    """What an int64 tensor takes: floats, numpy and tensor scalars, truth values; and what it refuses."""
    import numpy as np
    from evo_amd.ops import default_ops
    ops = default_ops()
    for tokens in ([3.0, 65], [np.int64(7), np.int32(-1)], [torch.tensor(9), torch.tensor(84, device="cuda")], [True, 67], [(1 << 63) - 1, -(1 << 63)]):
        ids = torch.zeros(5, 1, dtype=torch.int64, device="cuda")
        ops.put_tokens(ids, [4, np.int64(1)], tokens)
        assert ids[[4, 1], 0].tolist() == torch.tensor(tokens, dtype=torch.int64).tolist() and ids.count_nonzero().item() == 2
    ids = torch.zeros(5, 1, dtype=torch.int64, device="cuda")
    for slots, tokens in (([0], [1 << 63]), ([0], ["A"]), ([1.0], [5]), ([1 << 64], [5])):
        with pytest.raises((RuntimeError, TypeError, ValueError, OverflowError)):
            ops.put_tokens(ids, slots, tokens)
    assert not ids.any()


@pytest.mark.parametrize("n", [1, 256, 257])
def test_advance_positions(n):
    from evo_amd.ops import default_ops
    pos = torch.arange(n, device="cuda")
    default_ops().advance_positions(pos, 200)
    assert torch.equal(pos, (torch.arange(n, device="cuda") + 1).clamp(max=200))


@pytest.mark.parametrize("D", [1024, 4088, 4096, 8192])
@pytest.mark.parametrize("M", [1, 5, 16, 300])
def test_rmsnorm_rows_of_every_register_form(D, M):
    from evo_amd.ops import default_ops
    g = torch.Generator(device="cuda").manual_seed(D + M)
    x, s = torch.randn(M, D, device="cuda", generator=g).bfloat16(), torch.randn(D, device="cuda", generator=g).bfloat16()
    want = s.double() * (x.double() / (x.double().square().mean(1, keepdim=True).sqrt() + 1e-6))
    got = default_ops().rmsnorm(x, None, s, 1e-6)
    assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-6).all())      # one rounding, taken twice
