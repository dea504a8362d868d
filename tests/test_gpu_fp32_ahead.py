"""fp32 dense layers with the rows of x split ahead (csrc/gemm_f32_ahead.hip): every tile height, whole tiles and shares, remainders of rows and columns."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ahead(lib, x, w, bias=None):
    (M, K), N = x.shape, w.shape[0]
    plan = (ctypes.c_int64 * 6)()
    assert lib.evo_linear_f32_ahead_plan(M, N, K, ctypes.cast(plan, ctypes.c_void_p)) >= 0
    ws = torch.empty(plan[5], dtype=torch.uint8, device=DEV)
    y = torch.full((M, N), 7.0, device=DEV)
    rc = lib.evo_linear_f32_ahead(x.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), y.data_ptr(), M, N, K, ws.data_ptr(), plan[5],
                                  torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return y, list(plan)


@pytest.fixture(scope="module")
def lib():
    from evo_amd.ops import HipOps
    return HipOps().lib


# rows of a tile, whether tiles are taken whole, whether they are shared out
SIZES = [(17, 32, 256, 32, 1, 0), (17, 1056, 2048, 32, 0, 1), (161, 8224, 256, 48, 1, 0), (33, 1056, 2048, 48, 0, 1), (256, 8224, 256, 64, 1, 0), (63, 2080, 2048, 64, 0, 1),
         (513, 8224, 512, 80, 1, 0), (65, 2080, 2048, 80, 0, 1), (513, 8224, 256, 96, 1, 0), (81, 8224, 2048, 96, 0, 1), (640, 8224, 256, 112, 1, 0),
         (97, 2080, 2048, 112, 0, 1), (113, 8224, 2048, 128, 0, 1), (1151, 8224, 1056, 128, 1, 1)]


@pytest.mark.parametrize("M,N,K,rows,whole,shared", SIZES)
def test_sums_against_64_bits(lib, M, N, K, rows, whole, shared):
    """A large sum is rounded once in 32 k (at most 2^-23 of a partial sum for adders that cut, sqrt(K / 32) of it in the mean square), the parts left out are
    2^-27 of a product in the mean square; a few more roundings of 2^-24 where shares are added.  A row that is not finite leaves the others as they are."""
    g = torch.Generator().manual_seed(M + N)
    x, w, b = (torch.randn(*s, generator=g).to(DEV) for s in ((M, K), (N, K), (N,)))
    y, plan = ahead(lib, x, w, b)
    assert plan[0] == rows and (plan[2] > 0) == bool(whole) and (plan[4] > 0) == bool(shared)
    want = x.double() @ w.double().t() + b.double()
    assert ((y.double() - want).norm() / want.norm()).item() < 2.0 ** -23 * (K / 32) ** 0.5 + 2.0 ** -24
    assert ((y.double() - want).abs().max() / want.pow(2).mean().sqrt()).item() < 2e-5          # (no output left out)
    x[M // 2, K // 2] = float("nan")
    z, _ = ahead(lib, x, w, b)
    assert bool(torch.isnan(z[M // 2]).all())
    assert torch.equal(y[: M // 2], z[: M // 2]) and torch.equal(y[M // 2 + 1:], z[M // 2 + 1:])


@pytest.mark.parametrize("M,N,K", [(70, 256, 256), (129, 1056, 2048)])          # whole tiles, shares
@pytest.mark.parametrize("a,b", [(-74, -75), (-130, 40), (60, -145), (127, -30), (0, 0)])
def test_single_products_to_the_ends_of_the_range(lib, M, N, K, a, b):
    """One product per output, operands of 2^a and 2^b beside ordinary ones in other rows: 2^-24 + 2^-23 of the result and half the smallest value; exact zeros stay."""
    g = torch.Generator().manual_seed(11)
    x, w = (1 + torch.rand(M, K, generator=g)).double(), torch.zeros(N, K, dtype=torch.float64)
    at = torch.arange(N) % K
    w[torch.arange(N), at] = (1 + torch.rand(N, generator=g)).double()
    x[::3] *= 2.0 ** a
    w[::2] *= 2.0 ** b
    x[1::3, at[1]] = 0.0
    x, w = x.float(), w.float()
    want = x.double()[:, at] * w.double()[torch.arange(N), at]
    y = ahead(lib, x.to(DEV), w.to(DEV))[0].cpu().double()
    fits = want.abs() <= torch.finfo(torch.float32).max
    assert bool(((y - want).abs() <= want.abs() * (2.0 ** -24 + 2.0 ** -23 + 5 * 2.0 ** -30) + 2.0 ** -150)[fits].all())
    assert bool(torch.isinf(y[~fits & (want.abs() > 3.41e38)]).all())


@pytest.mark.parametrize("M,N,K", [(70, 512, 256), (70, 1056, 2048)])
def test_infinities_and_nan_as_in_a_plain_sum(lib, M, N, K):
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    x[3, 5], x[9, 0], w[17, 8], x[20, 8] = float("inf"), float("nan"), float("-inf"), 0.0
    x[31], w[33] = 0.0, 0.0
    y, want = ahead(lib, x.to(DEV), w.to(DEV))[0].cpu(), x @ w.t()
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    odd = torch.isinf(want)
    assert torch.equal(y[odd], want[odd]) and torch.isfinite(y[~odd & ~torch.isnan(want)]).all() and torch.equal(y == 0, want == 0)


def test_what_is_refused(lib):
    plan = (ctypes.c_int64 * 6)()
    p = ctypes.cast(plan, ctypes.c_void_p)
    assert lib.evo_linear_f32_ahead_plan(64, 100, 256, p) == -1 and lib.evo_linear_f32_ahead_plan(64, 128, 250, p) == -1
    assert lib.evo_linear_f32_ahead_plan(0xffff1, 256, 256, p) == -1
    assert lib.evo_linear_f32_ahead_plan(60000, 22016, 4096, p) == 0               # (over 1 GiB of workspace: the form that needs none)
    x, w = torch.zeros(64, 256, device=DEV), torch.zeros(256, 256, device=DEV)
    y = torch.empty(64, 256, device=DEV)
    assert lib.evo_linear_f32_ahead(x.data_ptr(), w.data_ptr(), None, y.data_ptr(), 64, 256, 256, None, 0, None) == -1
    assert lib.evo_linear_f32_ahead(x.data_ptr() + 4, w.data_ptr(), None, y.data_ptr(), 60, 256, 256, y.data_ptr(), 1 << 30, None) == -1
