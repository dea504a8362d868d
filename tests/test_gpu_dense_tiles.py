"""GPU parity of the dense layer's smaller tiles and parts of K (csrc/gemm_tile.hip) through the ops that take them.

Reference: the product of the bf16 operands in fp64, then what follows it, rounded once.  Tolerance: half a bf16 ulp of the result is 2^-9 of it, taken
twice; the fp32 sums add at most K 2^-24 of the sum of magnitudes, under 1e-3 for operands of unit variance and weights of variance 1 / K.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows on both sides of every tile's edge; columns and depths that lead to each tile, to parts of K, and to the persistent kernel
# (two launches one behind the other: test_two_launches)
SHAPES = [(65, 256, 64), (65, 4096, 4096), (127, 512, 1024), (129, 4096, 4096), (161, 12288, 512), (161, 4096, 11008), (255, 4096, 4096),
          (385, 4096, 4096), (513, 4096, 11008), (769, 4096, 4096), (770, 4096, 11008), (1023, 4096, 11008), (1024, 4096, 11008), (1537, 4096, 2048), (2048, 4096, 1088), (2049, 4096, 4096),
          (6400, 4096, 1024)]


def _ops():
    from evo_amd.ops import default_ops
    return default_ops()


def _data(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(M * 13 + N * 3 + K + seed)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).bfloat16()
    return g, x, w


def _close(got, want):
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + 1e-3).all()), f"max err {err.max().item():.3e}"


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("bias,res", [(False, False), (True, True)])
def test_plain(M, N, K, bias, res):
    ops = _ops()
    g, x, w = _data(M, N, K)
    b = torch.randn(N, device="cuda", generator=g).bfloat16() if bias else None
    buf = torch.randn(M + 8, N, device="cuda", generator=g).bfloat16()
    keep = buf.clone()
    want = x.double() @ w.double().T
    want = want if b is None else want + b.double()
    got = ops.linear_mfma(x, w, b, buf[:M] if res else None)
    _close(got, want + keep[:M].double() if res else want)
    assert torch.equal(buf[M:], keep[M:])                       # rows behind the last stay untouched
    again = ops.linear_mfma(x, w, b, keep[:M].clone() if res else None)
    assert torch.equal(got, again)                              # the parts are added in a fixed order


@pytest.mark.parametrize("M,N,K", [(65, 512, 1024), (161, 4096, 4096), (700, 16384, 512), (1537, 4096, 1024)])
@pytest.mark.parametrize("act,cols", [("silu", 256), ("gelu_tanh", 512), ("relu2", -1)])
def test_activation(M, N, K, act, cols):
    ops = _ops()
    g, x, w = _data(M, N, K, 1)
    cols = N if cols < 0 else cols
    z = x.double() @ w.double().T
    f = {"silu": torch.nn.functional.silu, "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh"), "relu2": lambda t: t.relu().square()}[act]
    want = torch.cat([f(z[:, :cols]), z[:, cols:]], 1)
    err = (ops.linear_act(x, w, act, cols).double() - want).abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + 4e-3).all())    # (the square's slope is up to 8 here, and v_rcp / v_exp add 2^-22 each)


@pytest.mark.parametrize("M,I,K", [(65, 128, 128), (100, 11008, 4096), (161, 11008, 4096), (255, 384, 1024), (300, 2048, 512), (513, 11008, 256), (1030, 2048, 4096)])
@pytest.mark.parametrize("order", ["plain", "grouped"])
@pytest.mark.parametrize("act", ["gelu", "silu"])
def test_gate(M, I, K, order, act):
    ops = _ops()
    g, x, w = _data(M, 2 * I, K, 2)
    z = (x.double() @ w.double().T).bfloat16().double()
    z1, z2 = z[:, :I], z[:, I:]
    want = (torch.nn.functional.gelu(z1) if act == "gelu" else torch.nn.functional.silu(z1)) * z2
    got = ops.mlp_gate(x, w if order == "plain" else None, w12g=None if order == "plain" else ops.pack_gate_weights(w), act=act)
    err = (got.double() - want).abs()
    # a value of z on the edge of two bf16 numbers may round the other way: 2^-8 of it, through a slope of at most 1.13 and the other factor
    assert bool((err <= want.abs() * 2.0 ** -7 + (z1.abs() + 0.2) * z2.abs() * 2.0 ** -7 + 1e-3).all()), err.max().item()


@pytest.mark.parametrize("B,T,N,K", [(1, 256, 768, 256), (1, 500, 12288, 4096), (2, 600, 12288, 1024), (3, 1000, 768, 4096)])
def test_transposed(B, T, N, K):
    ops = _ops()
    g, x, w = _data(B * T, N, K, 3)
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    xp = ops.rmsnorm_rows(x, torch.ones(K, device="cuda").bfloat16(), 1e-6, B, T)
    zt = ops.linear_t(xp, w, b, B, T)
    want = xp[: zt.shape[0] * 256].double() @ w.double().T + b.double()
    got = zt.permute(0, 2, 1).reshape(-1, N)
    _close(got, want)


@pytest.mark.parametrize("M,K", [(1024, 4096), (1536, 1024), (2304, 4096), (6400, 1024)])
def test_norm_folded(M, K):
    """Row factors in, sums of squares out, the blocked X: each against the same steps one by one."""
    ops = _ops()
    N = 4096
    g, x, w = _data(M, N, K, 4)
    res = torch.randn(M, N, device="cuda", generator=g).bfloat16()
    want = x.double() @ w.double().T + res.double()
    for blocked in (False, True):
        r = res.clone()
        if blocked:
            xb = x.view(M // 128, 128, K // 16, 16).permute(0, 2, 1, 3).contiguous()
            rstd = ops.linear_residual_yblk_stats_(r, xb, w, None, 1e-6)
        else:
            rstd = ops.linear_residual_stats_(r, x, w, None, 1e-6)
        _close(r, want)
        rms = r.double().square().mean(1).sqrt()
        assert bool(((rstd[:M].double() * (rms + 1e-6) - 1).abs() < 1e-5).all())
    w2 = (torch.randn(768, N, device="cuda", generator=g) / 64).bfloat16()
    _close(ops.linear_rs(r, rstd, w2, None, w2, torch.ones(N, device="cuda").bfloat16(), 1e-6), (r.double() / (rms + 1e-6)[:, None]) @ w2.double().T)
    gate = ops.mlp_gate_rs(r, rstd, ops.pack_gate_weights(w2[:512]), w2[:512], torch.ones(N, device="cuda").bfloat16(), 1e-6)
    z = ((r.double() / (rms + 1e-6)[:, None]) @ w2[:512].double().T).bfloat16().double()
    g_want = torch.nn.functional.gelu(z[:, :256]) * z[:, 256:]
    assert bool(((gate.double() - g_want).abs() <= g_want.abs() * 2.0 ** -7 + (z[:, :256].abs() + 0.2) * z[:, 256:].abs() * 2.0 ** -7 + 1e-3).all())


def test_without_a_workspace():
    """The same product, unsplit, when the caller has no room for the parts."""
    from evo_amd.ops import _stream
    ops = _ops()
    M, N, K = 161, 4096, 11008
    _, x, w = _data(M, N, K, 5)
    assert ops.lib.evo_dense_ws(0, 0, M, N, K) > 0
    y = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    assert ops.lib.evo_dense_bf16(0, 0, 0, x.data_ptr(), w.data_ptr(), None, None, y.data_ptr(), None, None, 0, M, N, K, 0, 0, 0, 0, None, 0, _stream()) == 0
    _close(y, x.double() @ w.double().T)


@pytest.mark.parametrize("M", [1024, 1100, 1536, 2304, 3000, 6400])
def test_same_bits_on_every_tile(M):
    """From 1,024 rows on a row's result does not depend on the tiles its batch runs on: the persistent kernel's own entries are the yardstick."""
    from evo_amd.ops import _stream
    ops, K = _ops(), 1024
    g, x, w = _data(M, 4096, K, 6)
    b = torch.randn(4096, device="cuda", generator=g).bfloat16()
    r = torch.randn(M, 4096, device="cuda", generator=g).bfloat16()
    rs = torch.rand((M + 255) // 256 * 256, device="cuda", generator=g) + 0.5
    p = lambda t: None if t is None else t.data_ptr()      # noqa: E731
    for bias, res, factor, stats in ((b, None, None, False), (b, r, None, False), (b, None, rs, False), (None, None, rs, False), (b, r, None, True)):
        want, got = (torch.empty(M, 4096, device="cuda", dtype=torch.bfloat16) if res is None else res.clone() for _ in range(2))
        ss = [torch.zeros(32, rs.numel(), device="cuda") for _ in range(2)] if stats else [None, None]
        assert ops.lib.evo_linear_mfma_nf_bf16(p(x), p(w), p(bias), None if res is None else p(want), p(want), p(factor), p(ss[0]), rs.numel() if stats else 0,
                                               M, 4096, K, _stream()) == 0
        ops._dense_layer(0, x, w, got, M, 4096, K, b=bias, res=None if res is None else got, rs=factor, ss=ss[1])
        assert torch.equal(got, want)
        assert not stats or torch.equal(ss[0][:, :M], ss[1][:, :M])
    for factor in (None, rs):
        want, got = (torch.empty(M, 2048, device="cuda", dtype=torch.bfloat16) for _ in range(2))
        if factor is None:
            assert ops.lib.evo_mlp_gate_mfma_bf16(p(x), p(w), p(want), M, 2048, K, 0, _stream()) == 0
        else:
            assert ops.lib.evo_mlp_gate_mfma_nf_bf16(p(x), p(rs), p(w), p(want), M, 2048, K, _stream()) == 0
        ops._dense_layer(1, x, w, got, M, 4096, K, rs=factor)
        assert torch.equal(got, want)


@pytest.mark.parametrize("M,tail", [(4700, (128, 128)), (5300, (192, 128)), (5700, (256, 128)), (8200, (64, 64)), (8500, (128, 64))])
def test_two_launches(M, tail):
    """Whole rounds of the persistent kernel, then the rest on each smaller tile: every form of the layer as above, the activation, the gate."""
    from evo_amd.ops import _stream
    from test_dense_plan import launches
    plan = launches(0, False, M, 4096, 1024)
    assert len(plan) == 2 and plan[0]["persistent"] and (plan[1]["tile_rows"], plan[1]["tile_cols"]) == tail
    assert M > 8000 or len(launches(0, True, M, 4096, 1024)) == 2
    assert M == 5700 or len(launches(1, False, M, 4096, 1024)) == 2
    test_same_bits_on_every_tile(M)
    ops = _ops()
    g, x, w = _data(M, 4096, 1024, 10)
    want, got = (torch.empty(M, 4096, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    assert ops.lib.evo_linear_act_mfma_bf16(x.data_ptr(), w.data_ptr(), None, want.data_ptr(), M, 4096, 1024, 2048, 1, _stream()) == 0
    ops._dense_layer(0, x, w, got, M, 4096, 1024, act=1, act_cols=2048)
    assert torch.equal(got, want)


@pytest.mark.parametrize("Mp,Tm", [(1024, 1024), (1536, 512), (2304, 768)])
def test_same_bits_transposed(Mp, Tm):
    from evo_amd.ops import _stream
    ops, N, K = _ops(), 12288, 512
    skip, rows = 1, Mp + Mp // Tm
    g, x, w = _data(rows, N, K, 7)
    b, rs = torch.randn(N, device="cuda", generator=g).bfloat16(), torch.rand(rows, device="cuda", generator=g) + 0.5
    want, got = (torch.empty(Mp // 256, N, 256, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    assert ops.lib.evo_linear_t_mfma_nf_bf16(x.data_ptr(), rs.data_ptr(), w.data_ptr(), b.data_ptr(), want.data_ptr(), Mp, N, K, rows, Tm, skip, _stream()) == 0
    ops._dense_layer(3, x, w, got, Mp, N, K, b=b, rs=rs, x_rows=rows, Tm=Tm, row_skip=skip)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,K", [(5249, 4096), (5300, 11008), (5376, 4096), (5376, 11008), (5631, 4096)])
def test_statistics_of_a_tail_launch(M, K):
    """Whole rounds of the persistent kernel, then a tail on smaller tiles whose last one overhangs the layer: the sums of squares are those of the persistent
    kernel in every strip, and nothing is written behind the last."""
    from evo_amd.ops import _stream
    from test_dense_plan import launches
    ops, N, ld = _ops(), 4096, (M + 255) // 256 * 256
    g, x, w = _data(M, N, K, 8)
    b, r = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((N,), (M, N)))
    plan = launches(0, True, M, N, K)
    assert M > 5376 or (len(plan) == 2 and plan[1]["first"] + -(-plan[1]["rows"] // plan[1]["tile_rows"]) * plan[1]["tile_rows"] > ld)
    want, got = r.clone(), r.clone()
    ss = [torch.full((N // 128 + 1, ld), -1.0, device="cuda") for _ in range(2)]      # one row more than the strips
    assert ops.lib.evo_linear_mfma_nf_bf16(x.data_ptr(), w.data_ptr(), b.data_ptr(), want.data_ptr(), want.data_ptr(), None, ss[0].data_ptr(), ld, M, N, K, _stream()) == 0
    ops._dense_layer(0, x, w, got, M, N, K, b=b, res=got, ss=ss[1][:-1])
    assert torch.equal(got, want)
    assert torch.equal(ss[0][:-1, :M], ss[1][:-1, :M]) and bool((ss[1][-1] == -1).all())
    if M % 128 == 0:
        blocked = r.clone()
        ss[1].fill_(-1.0)
        ops._dense_layer(0, x.view(M // 128, 128, K // 16, 16).permute(0, 2, 1, 3).contiguous(), w, blocked, M, N, K, xblk=1, b=b, res=blocked, ss=ss[1][:-1])
        assert torch.equal(blocked, want)
        assert torch.equal(ss[0][:-1, :M], ss[1][:-1, :M]) and bool((ss[1][-1] == -1).all())


def test_a_sequence_whose_layers_end_in_a_tail_launch():
    """One sequence of 5,300 tokens through four layers of width 4,096, norms folded and as passes of their own: two bf16 evaluations of one model."""
    from test_gpu_model import DEV, acgt, build
    from test_gpu_packed_prompts import WIDE
    _, _, m = build(WIDE)
    ids, was = acgt(1, 5299).to(DEV), m.ops.fuse_norm
    try:
        m.ops.fuse_norm = True
        folded = m(ids)[0].float()
        m.ops.fuse_norm = False
        plain = m(ids)[0].float()
    finally:
        m.ops.fuse_norm = was
    for rows in (slice(0, 64), slice(64, 4096), slice(4096, None)):
        assert ((folded[0, rows] - plain[0, rows]).norm() / plain[0, rows].norm()).item() < 3e-2


@pytest.mark.parametrize("N,Mp", [(1024, 4352), (1280, 3328), (4096, 1280)])
def test_transposed_last_tile_overhangs_the_weight(N, Mp):
    """Tiles of 192 weight rows, N no multiple of 192: the last tile's rows behind the weight have no bias."""
    from evo_amd.ops import _stream
    from test_dense_plan import launches
    ops, K = _ops(), 512
    assert N % 192 and [p["tile_cols"] for p in launches(3, False, Mp, N, K)] == [192]
    g, x, w = _data(Mp, N, K, 9)
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    want, got = (torch.zeros(Mp // 256, N, 256, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    assert ops.lib.evo_linear_t_mfma_bf16(x.data_ptr(), w.data_ptr(), b.data_ptr(), want.data_ptr(), Mp, N, K, _stream()) == 0
    ops._dense_layer(3, x, w, got, Mp, N, K, b=b)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,K,tile", [(65, 12288, 4096, (96, 48)), (96, 12288, 256, (96, 48)), (67, 11264, 1088, (96, 48)), (65, 22016, 4096, (96, 96)),
                                        (96, 20992, 512, (96, 96)), (129, 22016, 4096, (192, 96)), (161, 21760, 1088, (192, 96)), (192, 24576, 256, (192, 96))])
def test_tiles_of_odd_widths(M, N, K, tile):
    """Tiles of 96 and 48 columns: every epilogue, the last tile of a width that they do not divide, rows and columns behind the result untouched."""
    from evo_amd.ops import _stream
    import ctypes
    ops = _ops()
    gated = tile[1] == 96
    out = (ctypes.c_int64 * 14)()
    assert ops.lib.evo_dense_plan(int(gated), 0, M, N, K, ctypes.cast(out, ctypes.c_void_p)) == 1 and tuple(out[2:4]) == tile
    g, x, w = _data(M, N, K, 7)
    z = x.double() @ w.double().T
    rs = torch.rand(M, device="cuda", generator=g) + 0.5
    if gated:
        for order in (1, 2):
            wk = ops.pack_gate_weights(w) if order == 1 else w
            for act, f in ((0, torch.nn.functional.gelu), (1, torch.nn.functional.silu)):
                for scale in (None, rs) if act == 0 else (None,):
                    y = torch.full((M + 3, N // 2), 7.0, device="cuda", dtype=torch.bfloat16)
                    assert ops.lib.evo_dense_bf16(order, act, 0, x.data_ptr(), wk.data_ptr(), None, None, y.data_ptr(), None if scale is None else scale.data_ptr(), None, 0,
                                                  M, N, K, 0, 0, 0, 0, None, 0, _stream()) == 0
                    zz = (z if scale is None else z * scale.double()[:, None]).bfloat16().double()
                    z1, z2 = zz[:, :N // 2], zz[:, N // 2:]
                    want = f(z1) * z2
                    err = (y[:M].double() - want).abs()
                    assert bool((err <= want.abs() * 2.0 ** -7 + (z1.abs() + 0.2) * z2.abs() * 2.0 ** -7 + 1e-3).all()), err.max().item()      # (as test_gate)
                    assert bool((y[M:] == 7).all())
        return
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    r = torch.randn(M, N, device="cuda", generator=g).bfloat16()
    for bias, res, scale, act in ((0, 0, 0, 0), (1, 1, 0, 0), (1, 0, 1, 0), (0, 0, 1, 0), (1, 0, 0, 3)):
        y = torch.full((M + 3, N), 7.0, device="cuda", dtype=torch.bfloat16)
        assert ops.lib.evo_dense_bf16(0, act, 0, x.data_ptr(), w.data_ptr(), b.data_ptr() if bias else None, r.data_ptr() if res else None, y.data_ptr(),
                                      rs.data_ptr() if scale else None, None, 0, M, N, K, 256 if act else 0, 0, 0, 0, None, 0, _stream()) == 0
        want = (z * rs.double()[:, None] if scale else z) + (b.double() if bias else 0) + (r.double() if res else 0)
        if act:
            want = torch.cat([want[:, :256].relu().square(), want[:, 256:]], 1)
        err = (y[:M].double() - want).abs()
        assert bool((err <= want.abs() * 2.0 ** -8 + (4e-3 if act else 1e-3)).all()), err.max().item()                          # (as test_plain, test_activation)
        assert bool((y[M:] == 7).all())


def test_gate_on_a_weight_of_more_than_4_gib():
    """Tiles of 96 gated columns, the grouped weight's bytes more than 32 bits hold: every tile finds its rows (22,016 x 98,304; the tiles see 128 rows of it at a time)."""
    from evo_amd.ops import _stream
    import ctypes
    ops = _ops()
    M, N, K = 161, 22016, 98304
    out = (ctypes.c_int64 * 14)()
    assert ops.lib.evo_dense_plan(1, 0, M, N, K, ctypes.cast(out, ctypes.c_void_p)) == 1 and tuple(out[2:4]) == (192, 96)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = torch.empty(N // 64, 64, K, device="cuda", dtype=torch.bfloat16)          # (blocks of 32 rows of each half)
    for part in w.split(16):
        part.copy_(torch.randn(part.shape, device="cuda", generator=g) * K ** -0.5)
    y = torch.full((M, N // 2), 7.0, device="cuda", dtype=torch.bfloat16)
    assert ops.lib.evo_dense_bf16(1, 0, 0, x.data_ptr(), w.data_ptr(), None, None, y.data_ptr(), None, None, 0, M, N, K, 0, 0, 0, 0, None, 0, _stream()) == 0
    xd = x.double()
    for i, part in enumerate(w.split(8)):
        z = (xd @ part.reshape(-1, K).double().T).bfloat16().double().view(M, -1, 2, 32)
        z1, z2 = z[:, :, 0].reshape(M, -1), z[:, :, 1].reshape(M, -1)
        want, got = torch.nn.functional.gelu(z1) * z2, y[:, 256 * i:256 * i + z1.shape[1]].double()
        err = (got - want).abs()
        assert bool((err <= want.abs() * 2.0 ** -7 + (z1.abs() + 0.2) * z2.abs() * 2.0 ** -7 + 1e-3).all()), (i, err.max().item())             # (as test_gate)


@pytest.mark.parametrize("K", [2048, 2112])
@pytest.mark.parametrize("N", [16384, 12288])
def test_gate_either_side_of_the_staggered_starts(N, K):
    """Tiles in step up to 2,048 k and where halves of [W1; W2] lie a power of two apart, otherwise a k-step apart."""
    from evo_amd.ops import _stream
    ops = _ops()
    M = 65
    g, x, w = _data(M, N, K, 11)
    z = (x.double() @ w.double().T).bfloat16().double()
    z1, z2 = z[:, :N // 2], z[:, N // 2:]
    want = torch.nn.functional.gelu(z1) * z2
    for order in (1, 2):
        wk, y = ops.pack_gate_weights(w) if order == 1 else w, torch.full((M + 3, N // 2), 7.0, device="cuda", dtype=torch.bfloat16)
        assert ops.lib.evo_dense_bf16(order, 0, 0, x.data_ptr(), wk.data_ptr(), None, None, y.data_ptr(), None, None, 0, M, N, K, 0, 0, 0, 0, None, 0, _stream()) == 0
        err = (y[:M].double() - want).abs()
        assert bool((err <= want.abs() * 2.0 ** -7 + (z1.abs() + 0.2) * z2.abs() * 2.0 ** -7 + 1e-3).all()), err.max().item()              # (as test_gate)
        assert bool((y[M:] == 7).all())
