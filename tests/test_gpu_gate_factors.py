"""A gated layer whose rows have factors, with either gate, on every kernel that a size may lead to (csrc/gemm_tile.hip evo_dense_bf16, mode 1)."""
import pytest
import torch

from test_dense_plan import launches

pytestmark = pytest.mark.gpu


# tiles of 160, 192, 224 and 256 rows of the persistent kernel (sixteen rounds of it and more: x before the weights), smaller ones, both, parts of K
@pytest.mark.parametrize("M,N,K,rows", [(513, 11008, 2048, [160]), (801, 11008, 2048, [192]), (961, 11008, 2048, [224]), (1024, 11008, 1088, [256]), (24576, 11008, 256, [256]),
                                        (4700, 4096, 1024, [256, 128]), (600, 6912, 1024, None), (161, 4096, 2048, None)])
@pytest.mark.parametrize("act", [0, 1])
def test_gate_of_rows_with_factors(M, N, K, rows, act):
    from test_gpu_dense_tiles import _data, _ops
    plan = launches(1, False, M, N, K)
    assert [p["tile_rows"] for p in plan] == rows if rows else not any(p["persistent"] for p in plan)
    ops = _ops()
    g, x, w = _data(M, N, K, 13)
    rs = torch.rand((M + 255) // 256 * 256, device="cuda", generator=g) + 0.5
    got = torch.full((M + 8, N // 2), 7.0, device="cuda", dtype=torch.bfloat16)
    ops._dense_layer(1, x, w, got, M, N, K, act=act, rs=rs)
    for a in range(0, M, 4096):
        z = ((x[a:a + 4096].double() @ w.double().T) * rs[a:min(a + 4096, M), None].double()).bfloat16().double().view(-1, N // 64, 2, 32)
        z1, z2 = z[:, :, 0].reshape(-1, N // 2), z[:, :, 1].reshape(-1, N // 2)
        want = (torch.nn.functional.silu(z1) if act else torch.nn.functional.gelu(z1)) * z2
        err = (got[a:min(a + 4096, M)].double() - want).abs()
        # a value of z on the edge of two bf16 numbers may round the other way: 2^-8 of it, through a slope of at most 1.13 and the other factor
        assert bool((err <= want.abs() * 2.0 ** -7 + (z1.abs() + 0.2) * z2.abs() * 2.0 ** -7 + 1e-3).all()), err.max().item()
    assert bool((got[M:] == 7).all())
