"""fp32 decode attention, four waves a tile of 64 slots (csrc/latent.hip latent_decode_f32_kernel, csrc/heads.hip heads_decode_f32_kernel): every part against fp64 at
numbers of slots around a wave's 16 and a tile's 64.  Scores of up to 1,028 fp32 products are off by under 1,028 2^-24 of their terms' sum (below 1e-4 for these
operands), the probabilities by as much relatively; sums of at most 128 rows add 128 2^-24."""
import pytest
import torch

pytestmark = pytest.mark.gpu
USED = [1, 15, 16, 17, 63, 64, 65, 130, 192, 200]


def _check(part, ml, want_o, want_m, want_l, parts):
    """parts [B, n_split]: slots that each part has; one without slots is not looked at but for its empty denominator"""
    for b in range(part.shape[0]):
        for s in range(part.shape[2]):
            if parts[b][s] == 0:
                assert bool((ml[b, :, s, 1] == 0).all() and (part[b, :, s] == 0).all())
                continue
            assert bool(((ml[b, :, s, 0].double() - want_m[b, :, s]).abs() < 1e-4).all())
            f = torch.exp2(want_m[b, :, s] - ml[b, :, s, 0].double())                      # (the part's own maximum)
            assert bool(((ml[b, :, s, 1].double() / f / want_l[b, :, s] - 1).abs() < 2e-4).all())
            scale = want_o[b, :, s].norm(dim=-1)
            assert bool(((part[b, :, s].double() / f[:, None] - want_o[b, :, s]).norm(dim=-1) < 2e-4 * scale).all())


def _want(scores, values, n_split, used):
    """scores [B, H, slots] in log2 units (-inf: not seen), values [B, H, slots, dv] -> what each part keeps: slots [64 (split + n_split i), + 64)"""
    B, H, _ = scores.shape
    o, m, l = torch.zeros(B, H, n_split, values.shape[-1]).double().cuda(), torch.zeros(B, H, n_split).double().cuda(), torch.zeros(B, H, n_split).double().cuda()
    parts = [[0] * n_split for _ in range(B)]
    for b in range(B):
        for s in range(n_split):
            at = [u for u in range(used[b]) if u // 64 % n_split == s]
            at = [u for u in at if bool(torch.isfinite(scores[b, 0, u]))]
            parts[b][s] = len(at)
            if at:
                x = scores[b][:, at]
                m[b, :, s] = x.amax(1)
                p = torch.exp2(x - m[b, :, s, None])
                l[b, :, s], o[b, :, s] = p.sum(1), (p[..., None] * values[b][:, at]).sum(1)
    return o, m, l, parts


@pytest.mark.parametrize("R,dr,n_split,window", [(512, 64, 4, 256), (64, 32, 1, 256), (516, 4, 2, 256), (1024, 4, 3, 256), (128, 64, 2, 40)])
def test_latent(R, dr, n_split, window):
    from evo_amd.ops import _stream, default_ops
    B, H, ring, rs = len(USED), 3, 256, R + dr + 4
    g = torch.Generator(device="cuda").manual_seed(R)
    q, cache = torch.randn(B, H, rs, device="cuda", generator=g), torch.randn(B, ring, rs, device="cuda", generator=g)
    pos = torch.tensor([u - 1 for u in USED], device="cuda")
    part, ml = torch.full((B, H, n_split, R), 7.0, device="cuda"), torch.full((B, H, n_split, 2), 7.0, device="cuda")
    c = 0.5 / (R + dr) ** 0.5
    assert default_ops().lib.evo_latent_decode(q.data_ptr(), cache.data_ptr(), pos.data_ptr(), part.data_ptr(), ml.data_ptr(), B, H, R, dr, rs, ring, window, n_split, c, 1, 0, _stream()) == 0
    s = (q[..., :R + dr].double() @ cache[..., :R + dr].double().transpose(1, 2)) * c * 1.4426950408889634
    age = pos[:, None] - torch.arange(ring, device="cuda")
    s = s.masked_fill(((age < 0) | (age >= window))[:, None], float("-inf"))
    o, m, l, parts = _want(s, cache[:, None, :, :R].double().expand(B, H, ring, R), n_split, USED)
    _check(part, ml, o, m, l, parts)


@pytest.mark.parametrize("H,G,maps,dim,dv,n_split", [(4, 2, 1, 128, 128, 4), (2, 2, 2, 128, 256, 2), (3, 1, 1, 36, 4, 1), (2, 1, 1, 1028, 512, 3)])
def test_heads(H, G, maps, dim, dv, n_split):
    from evo_amd.ops import _stream, default_ops
    B, ring = len(USED), 256
    rs = G * (maps * dim + dv)
    ld = H * maps * dim + rs
    g = torch.Generator(device="cuda").manual_seed(dim)
    z, cache = torch.randn(B, ld, device="cuda", generator=g), torch.randn(B, ring, rs, device="cuda", generator=g)
    pos = torch.tensor([u - 1 for u in USED], device="cuda")
    part, ml = torch.full((B, H * maps, n_split, dv), 7.0, device="cuda"), torch.full((B, H * maps, n_split, 2), 7.0, device="cuda")
    c = 0.5 / dim ** 0.5
    assert default_ops().lib.evo_heads_decode(z.data_ptr(), ld, cache.data_ptr(), pos.data_ptr(), part.data_ptr(), ml.data_ptr(), B, H, G, maps, dim, dv, ring, rs, n_split, c, 1, 0, _stream()) == 0
    q = z[:, :H * maps * dim].double().view(B, H, maps, dim)
    k = cache[..., :G * maps * dim].double().view(B, ring, G, maps, dim).repeat_interleave(H // G, 2)
    v = cache[..., G * maps * dim:].double().view(B, ring, G, dv).repeat_interleave(H // G, 2)
    s = torch.einsum("bhmd,bthmd->bhmt", q, k).reshape(B, H * maps, ring) * c * 1.4426950408889634
    values = v.permute(0, 2, 1, 3).repeat_interleave(maps, 1)
    o, m, l, parts = _want(s, values, n_split, USED)
    for b, p in enumerate(parts):
        for i, n in enumerate(p):
            if n == 0:                                            # (the floor in the place of a maximum)
                part[b, :, i], ml[b, :, i, 1] = 0, 0
    _check(part, ml, o, m, l, parts)
