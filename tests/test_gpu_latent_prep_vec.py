"""Latent attention's preparation in 16-byte requests (csrc/latent.hip latent_prep_vec_kernel): more norm columns than a wave's first request, more rotated heads than its
threads, a shared key that is rotated in part, and sizes that stay element by element (test_gpu_mixers.py has the comparison and its tolerances)."""
import pytest
import torch
from test_gpu_mixers import TYPES, ops, test_latent_prep as compare  # noqa: F401

pytestmark = pytest.mark.gpu


@TYPES
@pytest.mark.parametrize("H,dn,dr,R,n_rot,ring", [(2, 8, 40, 1032, 16, 9), (70, 16, 64, 64, 64, 5), (1, 0, 16, 8, 16, 3), (2, 8, 16, 520, 8, 9), (3, 4, 16, 64, 16, 9)])
def test_sizes(ops, dt, H, dn, dr, R, n_rot, ring):  # noqa: F811
    compare(ops, dt, H, dn, dr, R, n_rot, ring)


@TYPES
@pytest.mark.parametrize("H,dn,dr,R,n_rot", [(32, 128, 64, 512, 64), (2, 8, 40, 1032, 16), (3, 16, 64, 264, 64), (1, 0, 16, 8, 16), (2, 8, 16, 520, 16)])
def test_the_bits_of_the_element_kernel(ops, dt, H, dn, dr, R, n_rot):  # noqa: F811
    """A row's norm and rotation are the same bits in 16-byte requests and element by element (the same rows one element behind an aligned address)."""
    from evo_amd.ops import _stream
    M, width = 1000, H * (dn + dr) + R + dr
    g = torch.Generator(device="cuda").manual_seed(R)
    rows, w = (torch.randn(*s, device="cuda", generator=g).to(dt) for s in ((M, width), (R,)))
    inv = 10000.0 ** (-torch.arange(0, n_rot, 2, device="cuda") / n_rot)
    pos = torch.arange(M, device="cuda") * 131 + 5
    out = []
    for off in (0, 1):
        ld = (width + 7) // 8 * 8 + off
        z = torch.zeros(M, ld, dtype=dt, device="cuda")
        z[:, :width] = rows
        c, kr, cache = (torch.full(s, 7.0, dtype=dt, device="cuda") for s in ((M, R), (M, dr), (M, 4, R + dr)))
        assert ops.lib.evo_latent_prep(z.data_ptr(), ld, c.data_ptr(), kr.data_ptr(), cache.data_ptr(), w.data_ptr(), inv.data_ptr(), pos.data_ptr(), None, None, M, H, dn, dr, R,
                                       n_rot, 4, R + dr, 1e-6, int(dt == torch.float32), _stream()) == 0
        out.append((z[:, :width], c, kr, cache))
    for a, b in zip(*out):
        assert torch.equal(a, b)


@TYPES
@pytest.mark.parametrize("B,H,dn,dr,R,n_rot,ring", [(1, 32, 128, 64, 512, 64, 1024), (2, 5, 16, 24, 64, 16, 7), (3, 2, 40, 72, 1032, 72, 9), (5, 3, 24, 200, 72, 130, 3),
                                                    (8, 32, 128, 64, 512, 64, 64), (13, 3, 200, 8, 520, 2, 40)])
def test_preparation_with_the_query_side(ops, dt, B, H, dn, dr, R, n_rot, ring):  # noqa: F811
    """latent_decode with `prep` against latent_prep in front of it: the same cached rows and the same result, bit for bit; queries as they were, other rows untouched."""
    from evo_amd.mixer_ops import MixerOps, TokenBatch
    g = torch.Generator(device="cuda").manual_seed(B)

    def rnd(*s):
        return torch.randn(*s, device="cuda", generator=g).to(dt)
    rs, dv, width = MixerOps.latent_row(R, dr), 24, H * (dn + dr) + R + dr
    qd, w, wuk, wuv, cache = rnd(B, (width + 7) // 8 * 8 + 8), rnd(R), rnd(H * dn, R), rnd(H * dv, R), rnd(B + 1, ring, rs)
    inv = 10000.0 ** (-torch.arange(0, n_rot, 2, device="cuda") / n_rot)
    sink, pos = torch.randn(H, device="cuda", generator=g), torch.arange(B, device="cuda") * 131 + 5
    sizes = (H, dn, dr, dv, R, ring, 0.05)
    if H * (dn + dr) % 8 or rs % 8:
        assert not ops.latent_prep_fits(qd, cache, w, inv, H, dn, dr, R)
        return
    assert ops.latent_prep_fits(qd, cache, w, inv, H, dn, dr, R)
    q2, c2, was = qd.clone(), cache.clone(), qd.clone()
    got = ops.latent_decode(qd, cache, pos, wuk, wuv, sink, *sizes, prep=(w, inv, 1e-6))
    ops.latent_prep(q2, H, dn, dr, R, w, inv, 1e-6, TokenBatch.of_decode(pos), c2, want_kv=False)
    want = ops.latent_decode(q2, c2, pos, wuk, wuv, sink, *sizes)
    assert torch.equal(qd, was) and torch.equal(cache, c2) and torch.equal(got, want)
