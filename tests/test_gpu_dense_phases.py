"""Tiles of 128 x 128, 192 x 96 and 96 x 96 whose operands come in phases (csrc/gemm_tile.hip PHASES): full last row tiles and ones a quarter short; below, and one row
fewer, the other inner loop.  128 x 128: sixteen k-steps and seventeen (K up to 2,048: above, tiles of fewer than 256 rows start a k-step apart and sum in another order), the
persistent kernel's bits in every form.  The narrow tiles: odd counts of k-steps, against fp64 sums.  Rows behind the last untouched."""
import pytest
import torch

from test_dense_launches import all_launches
from test_dense_plan import launches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [64, 320, 1024, 1088, 2048])
@pytest.mark.parametrize("M,N", [(223, 12288), (224, 12288), (256, 11008), (384, 6912), (481, 8192)])
def test_phases(M, N, K):
    from test_gpu_dense_tiles import _data, _ops
    from evo_amd.ops import _stream
    assert all([(p["tile_rows"], p["tile_cols"], p["parts"]) for p in launches(m, s, M, N, K)] == [(128, 128, 1)] for m, s in ((0, False), (0, True), (1, False)))
    assert all([p["slots"] for p in all_launches(m, s, False, M, N, K)] == [6 if K >= 1024 and M != 223 else 0] for m, s in ((0, False), (0, True), (1, False)))
    ops, ld = _ops(), (M + 255) // 256 * 256
    g, x, w = _data(M, N, K, 12)
    b, r = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((N,), (M, N)))
    rs = torch.rand(ld, device="cuda", generator=g) + 0.5

    def new():
        return torch.full((M + 8, N), 7.0, device="cuda", dtype=torch.bfloat16)
    if K < 128:                                                   # (one k-step: the persistent kernel wants two.  Half a bf16 ulp, and 64 fp32 sums)
        y = new()
        ops._dense_layer(0, x, w, y, M, N, K, b=b, res=r)
        want = x.double() @ w.double().T + b.double() + r.double()
        bound = want.abs() * 2.0 ** -8 + 64 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + b.double().abs() + r.double().abs())
        assert bool(((y[:M].double() - want).abs() <= bound).all()) and bool((y[M:] == 7).all())
        return
    for bias, res, scale, stats in ((None, None, None, False), (b, r, None, True), (b, None, rs, False)):
        got, want = new(), new()
        ss = [torch.full((N // 128 + 1, ld), -1.0, device="cuda") if stats else None for _ in range(2)]
        p = [None if t is None else t.data_ptr() for t in (bias, res, scale, ss[0])]
        assert ops.lib.evo_linear_mfma_nf_bf16(x.data_ptr(), w.data_ptr(), p[0], p[1], want.data_ptr(), p[2], p[3], ld if stats else 0, M, N, K, _stream()) == 0
        ops._dense_layer(0, x, w, got, M, N, K, b=bias, res=res, rs=scale, ss=ss[1][:-1] if stats else None)
        assert torch.equal(got, want) and bool((got[M:] == 7).all())
        if stats:
            assert torch.equal(ss[0][:-1, :M], ss[1][:-1, :M]) and bool((ss[1][-1] == -1).all())
    got, want = (torch.full((M + 8, N // 2), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    assert ops.lib.evo_mlp_gate_mfma_bf16(x.data_ptr(), w.data_ptr(), want.data_ptr(), M, N // 2, K, 0, _stream()) == 0
    ops._dense_layer(1, x, w, got, M, N, K)
    assert torch.equal(got, want) and bool((got[M:] == 7).all())


@pytest.mark.parametrize("M,N,K,tile,slots", [(80, 22016, 4096, 96, 8), (96, 20992, 4160, 96, 8), (79, 22016, 4096, 96, 0), (96, 20992, 4032, 96, 0),
                                              (192, 24576, 1024, 192, 5), (150, 22016, 1088, 192, 5), (149, 22016, 1088, 192, 0), (161, 21760, 960, 192, 0)])
def test_narrow_tiles(M, N, K, tile, slots):
    """96 gated columns: eight or five slots of w, first and last row of the ranges; one row or one k-step outside them the loop in turn."""
    from test_gpu_dense_tiles import test_tiles_of_odd_widths as compare
    for mode in (1, 2):
        assert [(p["tile_rows"], p["tile_cols"], p["parts"], p["slots"]) for p in all_launches(mode, False, False, M, N, K)] == [(tile, 96, 1, slots)]
    compare(M, N, K, (tile, 96))
