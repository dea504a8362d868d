"""The persistent dense kernel on tiles of 160, 192 and 224 rows (csrc/gemm_kernel.h, chosen by csrc/gemm_tile.hip): every form of the layer is bit for bit that of
256 rows, whose products are in the same order, and writes nothing beside its result."""
import pytest
import torch

from test_dense_plan import launches

pytestmark = pytest.mark.gpu
K = 2048


def _data(M, N, seed):
    from test_gpu_dense_tiles import _data
    return _data(M, N, K, seed)


def _rows(mode, M, N, stats=False):
    plan = launches(mode, stats, M, N, K)
    assert len(plan) == 1 and plan[0]["persistent"]
    return plan[0]["tile_cols" if mode == 3 else "tile_rows"]


# (one row into a tile and whole tiles; 16 and 24 columns of tiles)
@pytest.mark.parametrize("M,N,rows", [(2049, 4096, 160), (2080, 4096, 160), (1599, 6144, 160), (2561, 4096, 192), (2688, 4096, 192), (1729, 6144, 192), (3073, 4096, 224),
                                      (3136, 4096, 224), (1921, 6144, 224)])
def test_rows_by_columns(M, N, rows):
    from test_gpu_dense_tiles import _ops
    from evo_amd.ops import _stream
    ops, ld = _ops(), (M + 255) // 256 * 256
    assert _rows(0, M, N) == rows and _rows(0, M, N, True) == rows
    g, x, w = _data(M, N, 3)
    b, r = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((N,), (M, N)))
    rs = torch.rand(ld, device="cuda", generator=g) + 0.5
    for bias, res, scale, stats in ((None, None, None, 0), (b, None, None, 0), (b, r, None, 0), (None, r, None, 1), (b, r, None, 1), (b, None, rs, 0), (None, None, rs, 0)):
        out = []
        for short in (False, True):
            y = torch.full((M + 64, N), 7.0, device="cuda", dtype=torch.bfloat16)
            ss = torch.full((N // 128 + 1, ld), -1.0, device="cuda") if stats else None
            p = [None if t is None else t.data_ptr() for t in (bias, res, scale, ss)]
            if short:
                rc = ops.lib.evo_dense_bf16(0, 0, 0, x.data_ptr(), w.data_ptr(), p[0], p[1], y.data_ptr(), p[2], p[3], ld if stats else 0, M, N, K, 0, 0, 0, 0, None, 0, _stream())
            else:
                rc = ops.lib.evo_linear_mfma_nf_bf16(x.data_ptr(), w.data_ptr(), p[0], p[1], y.data_ptr(), p[2], p[3], ld if stats else 0, M, N, K, _stream())
            assert rc == 0
            out.append((y, ss))
        assert torch.equal(out[0][0], out[1][0]) and bool((out[1][0][M:] == 7).all())
        if stats:
            assert torch.equal(out[0][1][:-1, :M], out[1][1][:-1, :M]) and bool((out[1][1][-1] == -1).all())
    for act in (1, 2, 3):
        want, got = (torch.empty(M, N, device="cuda", dtype=torch.bfloat16) for _ in range(2))
        assert ops.lib.evo_linear_act_mfma_bf16(x.data_ptr(), w.data_ptr(), b.data_ptr() if act > 1 else None, want.data_ptr(), M, N, K, 1024, act, _stream()) == 0
        ops._dense_layer(0, x, w, got, M, N, K, act=act, act_cols=1024, b=b if act > 1 else None)
        assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,rows", [(513, 11008, 160), (640, 11008, 160), (801, 11008, 192), (960, 11008, 192), (961, 11008, 224), (1100, 11008, 224)])
def test_gated(M, N, rows):
    from test_gpu_dense_tiles import _ops
    from evo_amd.ops import _stream
    ops = _ops()
    assert _rows(1, M, N) == rows
    g, x, w = _data(M, N, 4)
    rs = torch.rand((M + 255) // 256 * 256, device="cuda", generator=g) + 0.5
    for act in (0, 1, None):
        want, got = (torch.full((M + 64, N // 2), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(2))
        if act is None:
            assert ops.lib.evo_mlp_gate_mfma_nf_bf16(x.data_ptr(), rs.data_ptr(), w.data_ptr(), want.data_ptr(), M, N // 2, K, _stream()) == 0
        else:
            assert ops.lib.evo_mlp_gate_mfma_bf16(x.data_ptr(), w.data_ptr(), want.data_ptr(), M, N // 2, K, act, _stream()) == 0
        ops._dense_layer(1, x, w, got, M, N, K, act=act or 0, rs=rs if act is None else None)
        assert torch.equal(got, want) and bool((got[M:] == 7).all())


# (12,288 and 6,144 rows of the weight: whole tiles of 192, half a tile more than whole ones of 160 and 224)
@pytest.mark.parametrize("Mp,N,rows,Tm", [(768, 12288, 160, 768), (1536, 6144, 160, 512), (1024, 12288, 192, 256), (2048, 6144, 192, 1024), (2304, 12288, 224, 768), (2304, 6144, 224, 2304)])
def test_transposed(Mp, N, rows, Tm):
    from test_gpu_dense_tiles import _ops
    from evo_amd.ops import _stream
    ops, skip = _ops(), 2
    assert _rows(3, Mp, N) == rows
    n = Mp + (Mp // Tm - 1) * skip
    g, x, w = _data(n, N, 5)
    b, rs = torch.randn(N, device="cuda", generator=g).bfloat16(), torch.rand(n, device="cuda", generator=g) + 0.5
    for bias in (None, b):
        for scale in (False, True):
            want, got = (torch.full((Mp // 256 + 1, N, 256), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(2))
            pb = None if bias is None else bias.data_ptr()
            if scale:
                assert ops.lib.evo_linear_t_mfma_nf_bf16(x.data_ptr(), rs.data_ptr(), w.data_ptr(), pb, want.data_ptr(), Mp, N, K, n, Tm, skip, _stream()) == 0
                ops._dense_layer(3, x, w, got, Mp, N, K, b=bias, rs=rs, x_rows=n, Tm=Tm, row_skip=skip)
            else:
                assert ops.lib.evo_linear_t_mfma_bf16(x.data_ptr(), w.data_ptr(), pb, want.data_ptr(), Mp, N, K, _stream()) == 0
                ops._dense_layer(3, x, w, got, Mp, N, K, b=bias)
            assert torch.equal(got, want) and bool((got[-1] == 7).all())


def test_against_fp32():
    """One size of each height against fp32 sums: the 256-row kernel's own bound, half a unit in the last place of bf16 and the sums' order."""
    from test_gpu_dense_tiles import _ops
    for M in (2100, 2600, 3200):
        g, x, w = _data(M, 4096, 6)
        y = torch.empty(M, 4096, device="cuda", dtype=torch.bfloat16)
        _ops()._dense_layer(0, x, w, y, M, 4096, K)
        want = x.double() @ w.double().T
        bound = want.abs() * 2.0 ** -8 + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        assert bool(((y.double() - want).abs() <= bound).all())
