"""Ungated layers of 65 to 255 rows on tiles that are one round of the chip, and in two parts where 128 x 64 would be (csrc/gemm_tile.hip tile_one_round)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,tile", [(97, 12288, 2048, (96, 96, 1, 0)), (160, 11264, 4096, (96, 96, 1, 0)), (161, 12288, 4096, (96, 96, 1, 8)), (192, 11264, 2112, (96, 96, 1, 8)),
                                        (97, 6144, 4096, (96, 48, 1, 0)), (192, 5632, 2048, (96, 48, 1, 0)), (193, 6144, 4096, (64, 96, 1, 0)), (255, 5632, 5120, (64, 96, 1, 0)),
                                        (65, 16384, 4096, (128, 128, 2, 0)), (128, 13824, 5120, (128, 128, 2, 0)), (240, 8192, 4096, (128, 128, 2, 0))])
def test_tiles_of_one_round(M, N, K, tile):
    """Every epilogue against the fp64 product, and the rows behind the result untouched.  Half a bf16 ulp is 2^-9 of a value, taken twice; fp32 sums add under 1e-3 (K 2^-24 of
    the sum of magnitudes), four times that behind a square."""
    from evo_amd.ops import _stream, default_ops
    ops = default_ops()
    out = (ctypes.c_int64 * 16)()
    assert ops.lib.evo_dense_launches(0, 0, 0, M, N, K, ctypes.cast(out, ctypes.c_void_p)) == 1 and (out[2], out[3], out[4], out[7]) == tile
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = torch.randn(M, K, device="cuda", generator=g).bfloat16(), (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).bfloat16()
    b, r = torch.randn(N, device="cuda", generator=g).bfloat16(), torch.randn(M, N, device="cuda", generator=g).bfloat16()
    rs = torch.rand(M, device="cuda", generator=g) + 0.5
    z = x.double() @ w.double().T
    n = ops.lib.evo_dense_ws(0, 0, M, N, K)
    ws = torch.empty(max(n, 16), dtype=torch.uint8, device="cuda")
    for bias, res, scale, act in ((0, 0, 0, 0), (1, 1, 0, 0), (1, 0, 1, 0), (0, 0, 1, 0), (1, 0, 0, 3)):
        y = torch.full((M + 3, N), 7.0, device="cuda", dtype=torch.bfloat16)
        assert ops.lib.evo_dense_bf16(0, act, 0, x.data_ptr(), w.data_ptr(), b.data_ptr() if bias else None, r.data_ptr() if res else None, y.data_ptr(),
                                      rs.data_ptr() if scale else None, None, 0, M, N, K, N if act else 0, 0, 0, 0, ws.data_ptr(), n, _stream()) == 0
        want = (z * rs.double()[:, None] if scale else z) + (b.double() if bias else 0) + (r.double() if res else 0)
        if act:
            want = want.relu().square()
        err = (y[:M].double() - want).abs()
        assert bool((err <= want.abs() * 2.0 ** -8 + (4e-3 if act else 1e-3)).all()), err.max().item()
        assert bool((y[M:] == 7).all())


@pytest.mark.parametrize("M,N,K", [(96, 12288, 1984), (97, 12288, 1984), (193, 12288, 4096), (161, 10240, 4096), (145, 6144, 6144), (128, 16384, 2048), (129, 16384, 4096)])
def test_what_stays(M, N, K):
    from evo_amd.ops import default_ops
    out = (ctypes.c_int64 * 16)()
    assert default_ops().lib.evo_dense_launches(0, 0, 0, M, N, K, ctypes.cast(out, ctypes.c_void_p)) == 1
    assert (out[2], out[3]) not in ((96, 96), (64, 96)) and (out[2], out[3], out[4]) != (128, 128, 2) and ((out[2], out[3]) != (96, 48) or M == 96)


@pytest.mark.parametrize("M,N,K,tile", [(97, 22016, 4096, (128, 96, 1, 7)), (112, 21760, 2112, (128, 96, 1, 7)), (128, 24576, 2048, (128, 96, 1, 7)), (97, 11264, 2048, (96, 96, 1, 0)),
                                        (128, 12288, 4096, (96, 96, 1, 0))])
def test_gated_tiles_of_one_round(M, N, K, tile):
    """Both gates on either order of the weight, with and without row factors.  A value of z on the edge of two bf16 numbers may round the other way: 2^-8 of it, through a slope of at
    most 1.13 and the other factor."""
    from evo_amd.ops import _stream, default_ops
    ops = default_ops()
    out = (ctypes.c_int64 * 16)()
    assert ops.lib.evo_dense_launches(1, 0, 0, M, N, K, ctypes.cast(out, ctypes.c_void_p)) == 1 and (out[2], out[3], out[4], out[7]) == tile
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = torch.randn(M, K, device="cuda", generator=g).bfloat16(), (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).bfloat16()
    rs = torch.rand(M, device="cuda", generator=g) + 0.5
    z = x.double() @ w.double().T
    for order, act, scale in ((1, 0, False), (2, 0, True), (1, 1, True), (2, 1, False)):
        wk, y = ops.pack_gate_weights(w) if order == 1 else w, torch.full((M + 3, N // 2), 7.0, device="cuda", dtype=torch.bfloat16)
        assert ops.lib.evo_dense_bf16(order, act, 0, x.data_ptr(), wk.data_ptr(), None, None, y.data_ptr(), rs.data_ptr() if scale else None, None, 0, M, N, K, 0, 0, 0, 0, None, 0,
                                      _stream()) == 0
        zz = (z * rs.double()[:, None] if scale else z).bfloat16().double()
        z1, z2 = zz[:, :N // 2], zz[:, N // 2:]
        want = (torch.nn.functional.silu(z1) if act else torch.nn.functional.gelu(z1)) * z2
        err = (y[:M].double() - want).abs()
        assert bool((err <= want.abs() * 2.0 ** -7 + (z1.abs() + 0.2) * z2.abs() * 2.0 ** -7 + 1e-3).all()), err.max().item()
        assert bool((y[M:] == 7).all())
