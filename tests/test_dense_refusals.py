"""What the dense layer's entry (csrc/gemm_tile.hip evo_dense_bf16) refuses before it launches anything."""
import pytest
import torch

from evo_amd import ops as evo_ops
from test_dense_plan import launches


@pytest.mark.skipif(torch.cuda.is_available(), reason="no memory behind the operands' addresses")
@pytest.mark.parametrize("Mp,N,K,rows", [(6400, 3072, 4096, 160), (6656, 3072, 4096, 192), (4608, 12288, 4096, 224), (5632, 3072, 4096, 0)])
def test_tokens_of_over_4_gib(Mp, N, K, rows):
    """Row factors of a transposed result: the token matrix's rows, those between its batch rows included, times K are below 4 GiB on the persistent kernel, whatever its tiles' height.
    (Without a GPU a call that is accepted ends in the launch's own error.)  The last size goes to smaller tiles instead, which have 64 bits."""
    plan, Tm = launches(3, False, Mp, N, K), 256
    assert [(p["tile_cols"], p["persistent"]) for p in plan] == [(rows or 160, 1)]

    def call(skip):
        n, p = Mp + (Mp // Tm - 1) * skip, 1 << 20
        return n * K * 2, evo_ops.load_library().evo_dense_bf16(3, 0, 0, p, p, None, None, p, p, None, 0, Mp, N, K, 0, n, Tm, skip, None, 0, None)
    skip = (0xffffffff // (2 * K) - Mp) // (Mp // Tm - 1)
    assert skip < 0x7fff
    below, rc = call(skip)
    assert below < 0xffffffff and rc not in (0, -1)
    over, rc = call(skip + 1)
    assert over >= 0xffffffff and (rc == -1 if rows else rc not in (0, -1))
