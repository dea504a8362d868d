"""GPU parity of the narrow weight-streaming layers at 5 to 32 rows (csrc/gemv.hip skinny_kw_kernel).  Reference: the product of the bf16 operands in
fp64, bias, residual and activation, one rounding.  Tolerance: twice half a bf16 ulp (2^-8 of the result) and 1e-3 for the fp32 sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows at the edges of 8, 16 and 32; one chunk of 128 k up to more chunks than waves and buffers hold; columns that end inside a workgroup's 16
@pytest.mark.parametrize("M", [5, 8, 9, 16, 17, 31, 32])
@pytest.mark.parametrize("N,K", [(16, 128), (40, 256), (512, 4096), (1000, 1152), (4096, 2176), (8191, 384), (264, 12288)])
@pytest.mark.parametrize("extra", [False, True])
def test_narrow_layer(M, N, K, extra):
    from evo_amd.ops import default_ops
    ops = default_ops()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).bfloat16()
    want = x.double() @ w.double().T
    if extra:
        b, r = torch.randn(N, device="cuda", generator=g).bfloat16(), torch.randn(M + 1, N, device="cuda", generator=g).bfloat16()
        keep, want = r.clone(), want + b.double()
        got = ops._linear_small_m(x, w, b, r[:M])
        want = want + keep[:M].double()
        assert got.data_ptr() == r.data_ptr() and torch.equal(r[M], keep[M])
    else:
        got, want = ops._linear_small_m(x, w, None, None, act=3), want.relu().square()
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + (1e-3 if extra else 4e-3)).all()), err.max().item()      # (the square's slope is up to 8)
