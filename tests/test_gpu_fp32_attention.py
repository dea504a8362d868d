"""The fp32 matrix-core form of prompt attention (csrc/window_attn.hip window_attn_f32_kernel) against the any-size kernel, which the tests of the heads
and of the latent mixer hold against fp64.  Tolerance: both sum up to 512 products and 300 weighted values in fp32, each within 2^-24 sqrt(n) of its own
sum, and exp of a score of up to 60 carries 60 x 2^-24: 2e-5 of the result's norm covers both."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def both(z, kv, kr, sink, H, G, maps, dn, dr, dv, window, keep, scale, lens, extra):
    from evo_amd.ops import default_ops
    ops = default_ops()
    cu = lambda ns: torch.tensor([0] + ns).cumsum(0).to(torch.int32).to(DEV)      # noqa: E731
    nk = G * maps * dn
    out = []
    for fast in (True, False):
        ops.mixer_mfma = fast
        try:
            out.append(ops._window_attn(z, kv[:, :nk], kv[:, nk:], kr, sink, H, G, maps, dn, dr, dv, window, keep, scale, 0.4, 0.7, 1e-4, cu(lens),
                                        cu([m + e for m, e in zip(lens, extra)]), max(lens)))
        finally:
            ops.mixer_mfma = True
    return out


# head dims at and between the instantiations' sizes, single-tile and many-tile windows, kept tokens before, at and behind a tile's edge
@pytest.mark.parametrize("H,G,maps,dn,dr,dv,window,keep,sink", [
    (2, 2, 1, 4, 0, 4, 1 << 29, 0, False), (4, 2, 1, 64, 0, 64, 1, 0, False), (2, 1, 1, 68, 0, 100, 31, 5, False), (3, 3, 1, 128, 64, 128, 64, 0, True),
    (2, 2, 1, 128, 64, 256, 33, 0, True), (2, 2, 1, 120, 72, 132, 1 << 29, 0, True), (2, 2, 1, 192, 64, 60, 100, 32, False), (2, 1, 2, 64, 0, 64, 1 << 29, 0, False),
    (2, 2, 2, 128, 0, 256, 70, 33, False), (4, 2, 2, 12, 0, 20, 32, 1, False)])
def test_matches_the_any_size_form(H, G, maps, dn, dr, dv, window, keep, sink):
    g = torch.Generator(device=DEV).manual_seed(dn + dv + window % 1000)
    lens, extra = [1, 2, 63, 64, 65, 129, 300], [0, 3, 5, 0, min(window - 1, 70), 0, 1]
    nq, nk, dq = sum(lens), sum(lens) + sum(extra), dn + dr
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)      # noqa: E731
    z, kv = rnd(nq, H * maps * dq + 4), rnd(nk, G * (maps * dn + dv))
    kv[::13, :G * maps * dn] *= 3.0                               # keys that stand out
    kr, s = (rnd(nk, dr) if dr else None), (rnd(H) if sink else None)
    fast, slow = both(z, kv, kr, s, H, G, maps, dn, dr, dv, window, keep, 1.0 / math.sqrt(dq), lens, extra)
    assert bool(torch.isfinite(fast).all())
    assert ((fast - slow).norm() / slow.norm()).item() < 2e-5


def test_scores_below_any_floor_and_infinite_values():
    """All scores of a row near -1e33, and an infinite value behind one key: what the any-size form gives, finite where that is."""
    T, n, dv = 70, 64, 64
    g = torch.Generator(device=DEV).manual_seed(3)
    q = torch.full((T, n), 1e16, device=DEV)
    k = -(1e16 + torch.rand(T, n, device=DEV, generator=g) * 1e9)
    v = torch.randn(T, dv, device=DEV, generator=g)
    v[40, 3] = float("inf")
    fast, slow = both(q, torch.cat([k, v], 1), None, None, 1, 1, 1, n, 0, dv, 1 << 29, 0, 1.0, [T], [0])
    assert torch.equal(torch.isfinite(fast), torch.isfinite(slow)) and bool(torch.isfinite(fast[:40]).all())
