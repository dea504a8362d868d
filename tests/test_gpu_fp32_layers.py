"""fp32 dense layers on the bf16 matrix cores (csrc/gemm_f32.hip): operands as three bf16 parts each."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from evo_amd.ops import HipOps
    o = HipOps()
    o._f32_layer_pays = lambda M, N, K: True                     # (the kernel itself, at sizes that the library would take too)
    return o


def rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


# a lone row tile and column tile, remainders of both, one k-step more than the parts of K divide (each tile and number of parts: PLANS below)
SHAPES = [(33, 256, 256), (63, 260, 288), (65, 512, 4096), (129, 1028, 1056), (300, 4096, 1024), (513, 260, 256), (1290, 2048, 512), (2049, 2052, 256), (4000, 4096, 256)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("bias", [False, True])
def test_no_further_from_64_bits_than_fp32(ops, M, N, K, bias):
    """Against the sum in 64 bits.  Each of the K / 16 x 6 matrix products adds to an fp32 sum: rounding of at most 2^-24 of a partial sum, which random
    walks to sqrt(K) of a product; the sum over the steps stays under 2^-24 sqrt(6 K / 16) in the mean square, doubled for the parts left out and for
    adders that cut."""
    x, w, b = rand(M, K, seed=1).to(DEV), rand(N, K, seed=2).to(DEV), rand(N, seed=3).to(DEV) if bias else None
    assert ops._f32_layer_ok(x, w, b)
    y = ops.linear(x, w, b)
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    err = ((y.double() - want).norm() / want.norm()).item()
    assert err < 2.0 ** -23 * (6 * K / 16) ** 0.5, err
    plain = torch.addmm(b, x, w.t()) if bias else x @ w.t()
    assert err < 1.25 * ((plain.double() - want).norm() / want.norm()).item() + 2.0 ** -24


def test_parts_are_exact_and_large_values_stay_finite(ops):
    """One product per output: x (times a power of two) comes back bit for bit, up to the largest fp32 value."""
    x = torch.cat([rand(40, 256, seed=4), rand(40, 256, seed=5) * 1e30, rand(40, 256, seed=6) * 1e-30]).to(DEV)
    x[0, 0], x[0, 1] = torch.finfo(torch.float32).max, -torch.finfo(torch.float32).max
    w = torch.zeros(256, 256, device=DEV)
    w[torch.arange(256), torch.randperm(256, generator=torch.Generator().manual_seed(7))] = 0.5
    assert torch.equal(ops.linear(x, w), x[:, w.argmax(1)] * 0.5)


# tile, parts of K: a size that takes them, remainders of rows and columns where that is one
PLANS = [((64, 64), 2, (657, 2044, 1024)), ((64, 64), 3, (257, 2048, 1056)), ((64, 128), 1, (642, 8196, 256)), ((64, 128), 4, (642, 2044, 1024)), ((64, 128), 8, (131, 4092, 4096)),
         ((128, 128), 1, (390, 8188, 256)), ((128, 128), 2, (775, 2044, 1024)), ((128, 128), 3, (517, 2044, 1024)), ((128, 128), 8, (69, 4092, 4096)),
         ((256, 256), 1, (1539, 8188, 256)), ((256, 256), 2, (1671, 4092, 4096)), ((256, 256), 8, (391, 4092, 4096))]


@pytest.mark.parametrize("tile,parts,shape", PLANS)
def test_every_tile_and_number_of_parts(ops, tile, parts, shape):
    """The bound above; a row that is not finite leaves the others bit for bit as they were."""
    M, N, K = shape
    out = (ctypes.c_int64 * 3)()
    assert ops.lib.evo_linear_f32_plan(M, N, K, ctypes.cast(out, ctypes.c_void_p)) == 0 and list(out) == [*tile, parts]
    test_no_further_from_64_bits_than_fp32(ops, M, N, K, True)
    x, w = rand(M, K, seed=14).to(DEV), rand(N, K, seed=15).to(DEV)
    y = ops.linear(x, w)
    x[M // 2, K // 2] = float("nan")
    z = ops.linear(x, w)
    assert bool(torch.isnan(z[M // 2]).all())
    assert torch.equal(y[: M // 2], z[: M // 2]) and torch.equal(y[M // 2 + 1:], z[M // 2 + 1:])


def test_a_lone_product(ops):
    """One product per output.  The parts left out are at most 2^-8 2^-17 of a product twice; of the six additions the last one's rounding counts, 2^-23 of
    the result for adders that cut (the others are of sums 2^-7 as large at most)."""
    g = torch.Generator().manual_seed(10)
    x, v = 1 + torch.rand(2048, 256, generator=g), 1 + torch.rand(256, generator=g)
    want = x.double() * v.double()
    err = ((ops.linear(x.to(DEV), torch.diag(v).to(DEV)).cpu().double() - want) / want).abs().max().item()
    assert err <= 2.0 ** -24 + 2.0 ** -23 + 5 * 2.0 ** -30, err


@pytest.mark.parametrize("M,N", [(70, 256), (390, 8192), (1540, 8192)])      # 64 x 64, 128 x 128, 256 x 256 tiles
@pytest.mark.parametrize("a,b", [(-70, -70), (-74, -75), (-110, 40), (-120, 100), (-130, 0), (-130, 40), (-145, 60), (60, -145), (-100, -30), (0, 0)])
def test_operands_and_results_near_the_smallest(ops, M, N, a, b):
    """One product per output, operands of 2^a and 2^b, beside columns of ordinary size in the other rows: what an fp32 multiplication gives, 2^-24 of the result
    and half the smallest value (or the lone product's 2^-22.4 where no part is near 2^-126)."""
    g = torch.Generator().manual_seed(11)
    K = 256
    x, w = (1 + torch.rand(M, K, generator=g)).double(), torch.zeros(N, K, dtype=torch.float64)
    at = torch.arange(N) % K
    w[torch.arange(N), at] = (1 + torch.rand(N, generator=g)).double()
    x[::3] *= 2.0 ** a
    w[::2] *= 2.0 ** b
    x[1::3, at[1]] = 0.0                                       # (an exact zero beside them)
    x, w = x.float(), w.float()
    want = x.double()[:, at] * w.double()[torch.arange(N), at]
    y = ops.linear(x.to(DEV), w.to(DEV)).cpu().double()
    assert bool(((y - want).abs() <= want.abs() * (2.0 ** -24 + 2.0 ** -23 + 5 * 2.0 ** -30) + 2.0 ** -150).all())


def test_rows_of_zeros(ops):
    x, w = rand(300, 512, seed=12).to(DEV), rand(516, 512, seed=13).to(DEV)
    x[7], x[100:200], w[3], w[260:300] = 0.0, 0.0, 0.0, 0.0
    y = ops.linear(x, w)
    want = x.double() @ w.double().t()
    assert torch.equal(y == 0, want == 0) and ((y.double() - want).norm() / want.norm()).item() < 1e-6
    assert not ops.linear(torch.zeros_like(x), w).any()


@pytest.mark.parametrize("K", [256, 4096])                     # one part of K, several
def test_infinities_and_nan(ops, K):
    x, w = rand(70, K, seed=8), rand(512, K, seed=9)
    x[3, 5] = float("inf")
    x[9, 0] = float("nan")
    w[17, 8] = float("-inf")
    x[20, 8] = 0.0
    # a sum over the largest value in any order, in one output only: elsewhere in that row no partial sum passes 3e38 (2 x 5e-3 + 4 sqrt(K) / 3e38)
    x[40, :2] = 3e38
    w[:, :2] *= 1e-3
    w[60, :2] = 3.0
    y, want = ops.linear(x.to(DEV), w.to(DEV)).cpu(), x @ w.t()
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    odd = torch.isinf(want)
    assert torch.equal(y[odd], want[odd]) and torch.isfinite(y[~odd & ~torch.isnan(want)]).all()


def test_what_keeps_torch(ops):
    x, w = rand(40, 256, seed=1).to(DEV), rand(256, 256, seed=2).to(DEV)
    assert ops._f32_layer_ok(x, w, None)
    assert not ops._f32_layer_ok(x[:32], w, None)              # few rows
    assert not ops._f32_layer_ok(x[:, :250].contiguous(), w[:, :250].contiguous(), None)
    assert not ops._f32_layer_ok(x.t().contiguous().t(), w, None)
    assert not ops._f32_layer_ok(torch.empty(40 * 256 + 1, device=DEV)[1:].view(40, 256), w, None)
    g = w.clone().requires_grad_()
    assert not ops._f32_layer_ok(x, g, None)
    ops.linear(x, g).sum().backward()
    assert torch.allclose(g.grad, x.sum(0).expand_as(g), rtol=1e-4, atol=1e-4)
    with torch.no_grad():
        assert ops._f32_layer_ok(x, g, None)
    with torch.autograd.forward_ad.dual_level():
        assert not ops._f32_layer_ok(x, w, None)


@pytest.mark.parametrize("M,N,K,own", [(33, 4096, 4096, False), (131, 4096, 4096, False), (132, 4096, 4096, True), (33, 22016, 4096, True), (329, 4096, 256, False), (330, 4096, 256, True),
                                       (32, 22016, 11008, False)])
def test_small_layers_are_the_librarys(M, N, K, own, monkeypatch):
    from evo_amd.ops import HipOps
    o, took = HipOps(), []
    monkeypatch.setattr(o, "_linear_f32", lambda x, w, b: took.append(x.shape) or torch.mm(x, w.t()))
    x, w = torch.zeros(M, K, device=DEV), torch.zeros(N, K, device=DEV)
    assert o.linear(x, w).shape == (M, N) and bool(took) == own


def test_tensors_of_another_device_keep_torch(ops, monkeypatch):
    x, w = rand(40, 256, seed=1).to(DEV), rand(256, 256, seed=2).to(DEV)
    assert ops._f32_layer_ok(x, w, None)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert not ops._f32_layer_ok(x, w, None)


@pytest.mark.filterwarnings("ignore")
def test_traces_counters_and_autocast_see_the_product(ops):
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    x, w = rand(40, 256, seed=1).to(DEV), rand(256, 256, seed=2).to(DEV)
    assert ops._f32_layer_ok(x, w, None)
    graph = make_fx(lambda a: ops.linear(a, w))(x)
    assert any("mm" in str(n.target) for n in graph.graph.nodes)
    assert torch.allclose(graph(2 * x), 2 * (x @ w.t()), rtol=1e-4, atol=1e-4)
    traced = torch.jit.trace(lambda a: ops.linear(a, w), x)
    assert torch.allclose(traced(2 * x), 2 * (x @ w.t()), rtol=1e-4, atol=1e-4)
    counter = FlopCounterMode(display=False)
    with counter:
        ops.linear(x, w)
    assert counter.get_total_flops() == 2 * 40 * 256 * 256
    with torch.autocast("cuda", torch.bfloat16):
        assert ops.linear(x, w).dtype == torch.bfloat16
    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    with Mode():
        ops.linear(x, w)
    assert torch.mm in seen
    with torch.device(DEV):                                      # a default device watches nothing
        assert ops._f32_layer_ok(x, w, None)


def test_under_capture(ops):
    x, w = rand(300, 1024, seed=1).to(DEV), rand(512, 1024, seed=2).to(DEV)
    want = ops.linear(x, w).clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        y = ops.linear(x, w)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        (x * 2).sum().item()
