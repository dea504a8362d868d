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


@TYPES
@pytest.mark.parametrize("B,H,dn,dr,dv,R,forms", [(8, 32, 128, 64, 128, 512, (4, 2, 2, 64)), (16, 32, 128, 64, 128, 512, (4, 4, 2, 128)), (7, 32, 128, 64, 100, 512, (4, 2, 2, 64)),
                                                  (16, 64, 24, 8, 24, 512, (4, 8, 4, 128)), (70, 64, 8, 8, 16, 256, (4, 8, 16, 128)), (2, 64, 16, 8, 128, 128, (2, 2, 2, 32))])
def test_decode_by_the_forms_of_its_maps(ops, dt, B, H, dn, dr, dv, R, forms):  # noqa: F811
    """Every form of the query side and of the value side, as evo_latent_forms names them, against windowed attention on uncompressed keys and values in 64 bits; with the
    preparation in the same launch the same bits."""
    import ctypes
    import math
    from evo_amd.mixer_ops import MixerOps, TokenBatch
    from oracle import vozalorn_ref as V
    out = (ctypes.c_int64 * 5)()
    assert ops.lib.evo_latent_forms(B, H, R, dv, 3, 0, ctypes.cast(out, ctypes.c_void_p)) == 0 and tuple(out)[:4] == forms
    g, ring, rs = torch.Generator().manual_seed(B), 20, MixerOps.latent_row(R, dr)

    def rnd(*s, scale=1.0):
        return (torch.randn(*s, generator=g) * scale).to(dt)
    width = H * (dn + dr) + R + dr
    cache, qd = rnd(B, ring, rs), rnd(B, (width + 7) // 8 * 8)
    cache[:, :, R + dr:] = 0.0
    wuk, wuv, w = rnd(H * dn, R, scale=1.5 / math.sqrt(R)), rnd(H * dv, R, scale=1 / math.sqrt(R)), rnd(R)
    sink, scale, pos = torch.randn(H, generator=g), 1.5 / math.sqrt(dn + dr), [3 * b % 50 for b in range(B)]
    inv = (10000.0 ** (-torch.arange(0, dr, 2) / dr)).cuda()
    at = torch.tensor(pos).cuda()
    dev = [t.cuda() for t in (wuk, wuv, sink)]
    sizes = (H, dn, dr, dv, R, ring, scale)
    # a token's own row as latent_prep makes it, and the queries as it leaves them
    q2, c2 = qd.cuda(), cache.cuda()
    ops.latent_prep(q2, H, dn, dr, R, w.cuda(), inv, 1e-6, TokenBatch.of_decode(at), c2, want_kv=False)
    q64, c64 = q2.cpu().double(), c2.cpu().double()
    for n_split in (1, 4, 5, 8, 9, 20):
        got = ops.latent_decode(q2, c2, at, *dev, *sizes, n_split=n_split)
        c3 = cache.cuda()
        assert torch.equal(got, ops.latent_decode(qd.cuda(), c3, at, *dev, *sizes, n_split=n_split, prep=(w.cuda(), inv, 1e-6))) and torch.equal(c3, c2)
        for b in {0, 1, B // 2, B - 1}:
            js = range(max(0, pos[b] - ring + 1), pos[b] + 1)
            rows = torch.stack([c64[b, j % ring, :R + dr] for j in js])
            k = torch.cat([(rows[:, :R] @ wuk.double().T).view(len(js), H, dn), rows[:, None, R:].expand(len(js), H, dr)], -1)
            v = (rows[:, :R] @ wuv.double().T).view(len(js), H, dv)
            want = V.windowed_sink_attention(q64[b:b + 1, :H * (dn + dr)].view(1, H, dn + dr), k, v, scale, ring, sink, torch.tensor([pos[b]]), torch.tensor(list(js))).reshape(1, -1)
            err = (got[b:b + 1].cpu().double() - want).norm() / want.norm()
            assert err < (2e-2 if dt == torch.bfloat16 else 1e-5), (b, n_split, float(err))       # (test_latent_decode's bounds)
