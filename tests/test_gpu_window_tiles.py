"""Prompt attention of the head sizes with tiles by DMA (csrc/window_attn.hip window_tile_kernel) against the any-size form in fp32 on the same bf16 values.
Tolerance: the probabilities and the result are rounded to bf16 (2^-9 each at most, independent): 4e-3 of the result's norm."""
import math

import pytest
import torch

from test_gpu_fp32_attention import both

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one block of queries and one more (256, with two maps 128), ragged last blocks and tiles, keys before the queries that are no whole tile, windows inside a
# tile, of whole tiles and wider than the prompt, kept tokens at, before and behind a tile's edge (and wider than the window's start), grouped heads, sinks
@pytest.mark.parametrize("H,G,maps,dr,dv,window,keep,sink", [
    (2, 2, 1, 64, 128, 1 << 29, 0, True), (3, 3, 1, 64, 128, 100, 0, True), (2, 2, 1, 64, 128, 64, 0, False), (4, 2, 1, 0, 128, 1 << 29, 0, False),
    (4, 1, 1, 0, 128, 129, 5, False), (2, 2, 1, 0, 128, 64, 64, True), (2, 1, 1, 0, 128, 90, 130, False), (2, 2, 1, 0, 128, 1, 0, False),
    (2, 2, 2, 0, 256, 1 << 29, 0, False), (4, 2, 2, 0, 256, 150, 0, False), (3, 1, 2, 0, 256, 17, 0, False)])
@pytest.mark.parametrize("lens,extra", [([129], [0]), ([256, 1, 257], [0, 0, 31]), ([300, 64, 2, 520], [5, 63, 0, 100])])
def test_matches_the_any_size_form(H, G, maps, dr, dv, window, keep, sink, lens, extra):
    g = torch.Generator(device=DEV).manual_seed(dr + dv + window % 1000 + lens[0])
    dn, nq, nk = 128, sum(lens), sum(lens) + sum(extra)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g).bfloat16()      # noqa: E731
    z, kv = rnd(nq, H * maps * (dn + dr) + 8), rnd(nk, G * (maps * dn + dv))
    kv[::13, :G * maps * dn] *= 4.0                               # keys that stand out: maxima that move late
    kr, s = (rnd(nk, dr) if dr else None), (torch.randn(H, device=DEV, generator=g) if sink else None)
    args = (s, H, G, maps, dn, dr, dv, window, keep, 1.0 / math.sqrt(dn + dr), lens, extra)
    fast = both(z, kv, kr, *args)[0].float()
    slow = both(z.float(), kv.float(), None if kr is None else kr.float(), *args)[1]
    assert bool(torch.isfinite(fast).all())
    err = (fast - slow).view(nq, H, dv).norm(dim=2) / slow.view(nq, H, dv).norm(dim=2).clamp_min(1e-3)
    assert err.max().item() < 4e-2 and ((fast - slow).norm() / slow.norm()).item() < 4e-3
    assert torch.equal(fast, both(z, kv, kr, *args)[0].float())


@pytest.mark.parametrize("H,G,maps,dr,dv", [(2, 2, 1, 64, 128), (2, 1, 1, 0, 128), (2, 2, 2, 0, 256)])
@pytest.mark.parametrize("past", [0, 5, 16, 40])
def test_an_infinite_value_stays_near_its_key(H, G, maps, dr, dv, past):
    """Queries before the tile of 64 keys that holds it, and those whose whole block of 32 (two maps: the whole tile) lies before it, stay finite."""
    g = torch.Generator(device=DEV).manual_seed(past)
    n, dn, at = 400, 128, 200
    z, kv = torch.randn(n, H * maps * (dn + dr), device=DEV, generator=g).bfloat16(), torch.randn(n + past, G * (maps * dn + dv), device=DEV, generator=g).bfloat16()
    kv[at, G * maps * dn:] = float("inf")
    kr = torch.randn(n + past, dr, device=DEV, generator=g).bfloat16() if dr else None
    fast = both(z, kv, kr, None, H, G, maps, dn, dr, dv, 1 << 29, 0, 0.08, [n], [past])[0]
    clean = at // 64 * 64 - past - (0 if maps == 2 else 31)        # (one map: a block of 32 queries that reaches the tile)
    assert bool(torch.isfinite(fast[:clean]).all()) and not bool(torch.isfinite(fast[at - past:]).any())


def test_negative_scale_and_short_prompts_take_the_other_kernels():
    g = torch.Generator(device=DEV).manual_seed(1)
    z, kv = torch.randn(200, 256, device=DEV, generator=g).bfloat16(), torch.randn(200, 512, device=DEV, generator=g).bfloat16()
    fast, slow = both(z, kv, None, None, 2, 2, 1, 128, 0, 128, 1 << 29, 0, -0.1, [200], [0])
    assert ((fast.float() - slow.float()).norm() / slow.float().norm()).item() < 8e-3
    fast, slow = both(z[:100], kv[:100], None, None, 2, 2, 1, 128, 0, 128, 1 << 29, 0, 0.1, [100], [0])
    assert ((fast.float() - slow.float()).norm() / slow.float().norm()).item() < 8e-3


@pytest.mark.parametrize("dr,keep", [(64, 0), (0, 0), (0, 5)])
def test_a_sink_that_is_not_finite(dr, keep):
    """NaN: that head's outputs are; -inf: no sink; +inf: all weight is the sink's."""
    H, dn, dv, n = 4, 128, 128, 200
    g = torch.Generator(device=DEV).manual_seed(dr + keep)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g).bfloat16()      # noqa: E731
    z, kv, kr = rnd(n, H * (dn + dr)), rnd(n, H * (dn + dv)), (rnd(n, dr) if dr else None)
    run = lambda s: both(z, kv, kr, s, H, H, 1, dn, dr, dv, 150, keep, 0.08, [n], [0])[0].view(n, H, dv)      # noqa: E731
    plain = run(None)
    got = run(torch.tensor([float("nan"), -math.inf, math.inf, -math.inf], device=DEV))
    assert bool(torch.isnan(got[:, 0]).all()) and not got[:, 2].any()
    assert torch.equal(got[:, 1], plain[:, 1]) and torch.equal(got[:, 3], plain[:, 3])
