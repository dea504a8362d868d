"""GPU parity of the weight-streaming layers whose operands reach LDS by asynchronous loads (csrc/gemv.hip skinny_ring_kernel).  Reference: the product of the bf16
operands in fp64, bias, residual and activation, one rounding.  Tolerance: twice half a bf16 ulp (2^-8 of the result) and 1e-3 for the fp32 sums of up to
12,288 products of variance 1 / K.  Rows behind the operands' ends hold NaN: nothing of them may reach a result."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _framed(rows, cols, g, scale=1.0):
    """[rows, cols] bf16, 64 rows of NaN behind it in the same buffer."""
    t = torch.full((rows + 64, cols), float("nan"), device=DEV, dtype=torch.bfloat16)
    t[:rows] = (torch.randn(rows, cols, device=DEV, generator=g) * scale).bfloat16()
    return t[:rows]


# rows at the edges of 16, 32 and 64; columns that leave unequal and odd shares on 256 workgroups, every number of waves, two rounds; one chunk of 128 k, fewer
# than stages, more than starts.  The last three: parts of K
@pytest.mark.parametrize("M", [3, 5, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(4097, 128), (8191, 384), (8192, 4096), (12289, 256), (16386, 640), (22016, 4224), (24577, 384), (4096, 8192), (1024, 12288), (2048, 1152)])
@pytest.mark.parametrize("extra", [False, True])
def test_linear(M, N, K, extra):
    from evo_amd.ops import default_ops
    ops = default_ops()
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = _framed(M, K, g), _framed(N, K, g, K ** -0.5)
    want = x.double() @ w.double().T
    if extra:
        b, r = torch.randn(N, device=DEV, generator=g).bfloat16(), torch.randn(M + 1, N, device=DEV, generator=g).bfloat16()
        keep, want = r.clone(), want + b.double()
        got, want = ops._linear_small_m(x, w, b, r[:M]), want + keep[:M].double()
        assert got.data_ptr() == r.data_ptr() and torch.equal(r[M], keep[M])
    else:
        got, want = ops._linear_small_m(x, w, None, None, act=3), want.relu().square()
    assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + (1e-3 if extra else 4e-3)).all())        # (the square's slope is up to 8)


# several rounds of workgroups, of three and of four waves; parts of K on 4,097 to 8,192 columns, and the sizes around them that take one sum
@pytest.mark.parametrize("M", [5, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K,few,many", [(24578, 256, 0, 0), (33024, 640, 0, 0), (50304, 384, 0, 0), (4160, 8192, 3, 3), (5120, 4096, 0, 3), (5504, 8192, 0, 2), (6912, 4224, 0, 2),
                                          (8192, 8320, 0, 2), (8192, 4224, 0, 0), (6912, 3968, 0, 0), (3072, 8320, 5, 5), (8256, 8192, 0, 0)])
def test_linear_in_rounds_and_parts(M, N, K, few, many):
    from evo_amd.ops import default_ops
    ops = default_ops()
    assert ops.lib.evo_linear_parts(M, N, K) == (0 if M < 17 else few if M <= 32 else many)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = _framed(M, K, g), _framed(N, K, g, K ** -0.5)
    b, r = torch.randn(N, device=DEV, generator=g).bfloat16(), torch.randn(M + 1, N, device=DEV, generator=g).bfloat16()
    keep = r.clone()
    got, want = ops._linear_small_m(x, w, b, r[:M]), x.double() @ w.double().T + b.double() + keep[:M].double()
    assert torch.equal(r[M], keep[M]) and bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-3).all())


# a workgroup per CU on 4,097 to 7,680 columns: shares of 16 and 17, 28, 29 and 30 columns, stages that outnumber nothing, chunks that are few against the starts; the sizes beside
@pytest.mark.parametrize("M", [5, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(4097, 2048), (4112, 2176), (7168, 2048), (7169, 2048), (7169, 4096), (7680, 4096), (7681, 4096), (6721, 1920)])
def test_linear_spread(M, N, K):
    test_linear(M, N, K, True)


@pytest.mark.parametrize("M", [5, 16, 17, 64])
@pytest.mark.parametrize("I,K", [(2064, 2048), (2080, 4096), (3584, 2048), (3616, 4096), (3840, 4096)])
def test_gate_spread(M, I, K):
    test_gate(M, I, K, I % 32 == 0)


@pytest.mark.parametrize("M", [3, 5, 16, 17, 33, 64])
@pytest.mark.parametrize("I,K", [(32, 128), (96, 384), (2080, 256), (5504, 1152), (8224, 2176), (12320, 1408), (16416, 256)])
@pytest.mark.parametrize("grouped", [False, True])
def test_gate(M, I, K, grouped):
    from evo_amd.ops import default_ops
    ops = default_ops()
    g = torch.Generator(device=DEV).manual_seed(M + I + K)
    x, w = _framed(M, K, g), _framed(2 * I, K, g, 1.5 * K ** -0.5)
    packed = None
    if grouped:
        packed = _framed(2 * I, K, g)
        packed.copy_(ops.pack_gate_weights(w.contiguous()))
    for act in ("gelu", "silu"):
        got = ops.mlp_gate(x, None if grouped else w, w12g=packed, act=act)
        z = (x.double() @ w.double().T).float().bfloat16().double()
        u, v = z[:, :I], z[:, I:]
        want = (torch.nn.functional.gelu(u) if act == "gelu" else torch.nn.functional.silu(u)) * v
        # (a product whose sum lies between two bf16 values may round to the other one: 2^-8 of it, and the gate's slope is at most 1.13)
        assert got.shape == (M, I) and bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -6 + 2e-3 * want.abs().max()).all())
        assert ((got.double() - want).norm() / want.norm()).item() < 4e-3


@pytest.mark.parametrize("I,K,M,names", [(1024, 2176, 8, 2), (2048, 3072, 64, 2), (256, 8192, 32, 2), (1376, 8320, 17, 2), (256, 4096, 33, 1), (1024, 2048, 8, 1),
                                         (1024, 2944, 33, 1), (2080, 4096, 8, 1), (1024, 4096, 4, 1)])
@pytest.mark.parametrize("grouped", [False, True])
def test_gate_of_narrow_layers(I, K, M, names, grouped):
    """Up to 2,048 gated columns of long rows: the layer and the gate in a launch each; regrouped weights from K = 8,192 on."""
    from evo_amd.ops import default_ops
    ops = default_ops()
    g = torch.Generator(device=DEV).manual_seed(M + I + K)
    x, w = _framed(M, K, g), _framed(2 * I, K, g, 1.5 * K ** -0.5).contiguous()
    ran, real = [], ops._t
    ops._t = lambda name: (ran.append(name), real(name))[1]
    try:
        wg = ops.pack_gate_weights(w) if grouped else None
        got, plain = ops.mlp_gate(x, None if grouped else w, w12g=wg), ran[:]
        scale = torch.rand(K, generator=g, device=DEV).bfloat16() + 0.5
        normed, want_n = ops.mlp_gate(x, None if grouped else w, scale, 1e-6, w12g=wg), ops.mlp_gate(ops.rmsnorm(x, None, scale, 1e-6), None if grouped else w, w12g=wg)
    finally:
        del ops._t
    assert M < 5 or torch.equal(normed, want_n)
    assert plain == (["gemv", "gelu_gate"] if names == 2 and (not grouped or K >= 8192) else ["gemv_gate"])
    z = (x.double() @ w.double().T).float().bfloat16().double()
    want = torch.nn.functional.gelu(z[:, :I]) * z[:, I:]
    assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -6 + 2e-3 * want.abs().max()).all())            # (as test_gate)
    assert ((got.double() - want).norm() / want.norm()).item() < 4e-3


def test_rows_off_16_bytes():
    """Operands that the asynchronous loads can't take keep the other forms."""
    from evo_amd.ops import default_ops
    ops = default_ops()
    g = torch.Generator(device=DEV).manual_seed(1)
    M, N, K = 8, 8192, 512
    x = torch.randn(M * K + 4, device=DEV, generator=g).bfloat16()[4:].view(M, K)
    w = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    want = x.double() @ w.double().T
    assert bool(((ops.linear(x, w).double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-3).all())
    u, v = want.float().bfloat16().double().split(N // 2, 1)
    gate = torch.nn.functional.gelu(u) * v
    assert ((ops.mlp_gate(x, w).double() - gate).norm() / gate.norm()).item() < 4e-3
    assert torch.equal(ops.mlp_gate(x, None, w12g=ops.pack_gate_weights(w)), ops.mlp_gate(x.clone(), w))     # (copied to a place that they can)


# layers of up to 4,096 columns at 3 to 32 rows: bias and residual four values a request, and one (odd columns, addresses two bytes on), each without the other
@pytest.mark.parametrize("M", [3, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(4096, 2048), (4094, 2048), (2052, 2176), (2049, 4096), (516, 1024), (20, 256)])
@pytest.mark.parametrize("odd", [0, 1])
def test_narrow_epilogue(M, N, K, odd):
    from evo_amd.ops import default_ops
    ops = default_ops()
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = _framed(M, K, g), _framed(N, K, g, K ** -0.5)
    plain = x.double() @ w.double().T
    b = torch.randn(N + 1, device=DEV, generator=g).bfloat16()[odd:odd + N]
    for bias in (None, b):
        for with_res in (False, True):
            if not with_res and bias is None:
                continue
            r = torch.randn(M * N + N + 1, device=DEV, generator=g).bfloat16()
            keep, res = r.clone(), r[odd:odd + M * N].view(M, N) if with_res else None
            want = plain + (0 if bias is None else bias.double()) + (keep[odd:odd + M * N].view(M, N).double() if with_res else 0)
            got = ops._linear_small_m(x, w, bias, res)
            assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-3).all())
            if with_res:
                assert got.data_ptr() == res.data_ptr() and torch.equal(r[odd + M * N:], keep[odd + M * N:]) and torch.equal(r[:odd], keep[:odd])
