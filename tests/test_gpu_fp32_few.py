"""fp32 dense layers of one to four rows (csrc/gemv_f32.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from evo_amd.ops import HipOps
    return HipOps()


# requests a row (eighths of K of 256 values): one with a single lane, whole, and a few lanes more, up to eight; rows per workgroup from one to the most
# (131,076 rows of K = 32: 512, and more workgroups than CUs), fewer rows than CUs
SIZES = [(1, 32), (131076, 32), (255, 2048), (257, 2080), (1030, 4096), (300, 4128), (777, 6144), (513, 8192), (300, 8224), (333, 11008), (290, 12288), (270, 14336), (259, 16384)]


@pytest.mark.parametrize("N,K", SIZES)
@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_sums_against_64_bits(ops, M, N, K):
    """A lane adds at most 32 products one after the other, ten additions join 512 lanes' sums and the bias: under 2^-24 sqrt(32 + 10) in the mean square of sums of
    K random products, sqrt(K) in the mean square (a lone sum may cancel: its error is held against that too), 2^-20 for the largest."""
    g = torch.Generator().manual_seed(N + K + M)
    x, w, b = (torch.randn(*s, generator=g).to(DEV) for s in ((M, K), (N, K), (N,)))
    assert ops._f32_few_ok(x, w, b)
    for bias in (b, None):
        y = ops.linear(x, w, bias)
        want = x.double() @ w.double().t() + (0 if bias is None else bias.double())
        assert y.shape == (M, N) and ((y.double() - want).norm() / (K * M * N) ** 0.5).item() < 2.0 ** -24 * 42 ** 0.5
        assert ((y.double() - want).abs().max() / K ** 0.5).item() < 2.0 ** -20


@pytest.mark.parametrize("K", [2080, 4096])
def test_not_finite(ops, K):
    """Lanes that the last request does not reach take no part: an infinity or NaN stays in its row of w and of x."""
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(3, K, generator=g), torch.randn(40, K, generator=g)
    w[5, K - 1], w[9, 0], x[2, 7] = float("inf"), float("nan"), float("-inf")
    x[1] = 0.0
    want = x @ w.t()
    y = ops.linear(x.to(DEV), w.to(DEV)).cpu()
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(y[torch.isinf(want)], want[torch.isinf(want)])
    assert torch.isfinite(y[torch.isfinite(want)]).all() and torch.equal(y == 0, want == 0)


def test_what_keeps_torch(ops, monkeypatch):
    took = []
    monkeypatch.setattr(ops, "_linear_few_f32", lambda x, w, b: took.append(x.shape) or torch.mm(x, w.t()))
    x, w = torch.randn(5, 256, device=DEV), torch.randn(64, 256, device=DEV)
    ops.linear(x, w)                                             # five rows
    ops.linear(x[:2, :250].contiguous(), w[:, :250].contiguous())
    ops.linear(x[:, :128][:2], w[:, :128].contiguous())          # strides
    ops.linear(torch.empty(513, device=DEV)[1:].view(2, 256), w)
    ops.linear(x[:2], w.clone().requires_grad_())
    with torch.autocast("cuda", torch.bfloat16):
        ops.linear(x[:2], w)
    assert not took
    ops.linear(x[:2], w)
    assert took == [(2, 256)]


def test_under_capture(ops):
    x, w = torch.randn(3, 1024, device=DEV), torch.randn(700, 1024, device=DEV)
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
