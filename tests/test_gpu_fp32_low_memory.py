"""fp32 dense layers where the card has no room for the parts of x (csrc/gemm_f32_ahead.hip): the form without a workspace, as before that kernel came."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_no_room_for_the_parts_of_x():
    from evo_amd.ops import HipOps, _stream
    ops, (M, N, K) = HipOps(), (4000, 4096, 4096)
    plan = (ctypes.c_int64 * 6)()
    assert ops.lib.evo_linear_f32_ahead_plan(M, N, K, ctypes.cast(plan, ctypes.c_void_p)) == 1 and ops.lib.evo_linear_f32_ws(M, N, K) == 0
    g = torch.Generator(device=DEV).manual_seed(3)
    x, w, b = (torch.randn(*s, device=DEV, generator=g) for s in ((M, K), (N, K), (N,)))
    want = torch.empty(M, N, device=DEV)
    assert ops.lib.evo_linear_f32(x.data_ptr(), w.data_ptr(), b.data_ptr(), want.data_ptr(), M, N, K, None, 0, _stream()) == 0
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + 4 * M * N + (8 << 20)           # the result and 8 MiB; the parts are 94
    assert plan[5] > 90 << 20
    try:
        torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(0).total_memory, 0)
        with torch.inference_mode():
            got = ops.linear(x, w, b)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, 0)
    assert torch.equal(got, want)
