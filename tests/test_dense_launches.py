"""The launches of a dense layer as csrc/gemm_tile.hip makes them (evo_dense_launches, on the host): blocked x, and which of the two inner loops a tile runs."""
import ctypes

import pytest

from evo_amd import ops as evo_ops
from test_dense_plan import KEYS, launches


def all_launches(mode, stats, xblk, M, N, K):
    out = (ctypes.c_int64 * 16)()
    n = evo_ops.load_library().evo_dense_launches(mode, int(stats), int(xblk), M, N, K, ctypes.cast(out, ctypes.c_void_p))
    assert n in (1, 2), n
    return [dict(zip(KEYS + ("slots",), out[8 * i:8 * i + 8])) for i in range(n)]


@pytest.mark.parametrize("N,K", [(4096, 4096), (4096, 11008), (4096, 10944), (2048, 2048), (1024, 1024), (5120, 5120), (768, 768)])
def test_blocked_statistics_stay_in_their_strip(N, K):
    """Blocked x: never on tiles of 160 to 224 rows (its blocks of 128 rows lie whole in a tile), every row's statistic and nothing of the next strip."""
    other = 0
    for M in range(256, 12001, 256):
        end, plan = 0, all_launches(0, True, True, M, N, K)
        for p in plan:
            assert p["first"] == end and p["rows"] > 0 and p["slots"] == 0 and (not p["persistent"] or p["tile_rows"] == 256)
            end += p["rows"]
            assert end <= p["stat_end"] <= M
        assert end == M
        other += [p["tile_rows"] for p in plan] != [p["tile_rows"] for p in launches(0, True, M, N, K)]
    assert other > 0 or K < 2048


def test_the_short_form():
    lib, out = evo_ops.load_library(), (ctypes.c_int64 * 16)()
    for M in list(range(65, 300)) + [513, 2304, 4700, 9000]:
        for mode, stats in ((0, 0), (0, 1), (1, 0), (2, 0)):
            assert [[p[k] for k in KEYS] for p in all_launches(mode, stats, False, M, 8192, 2048)] == [[p[k] for k in KEYS] for p in launches(mode, stats, M, 8192, 2048)]
    p = ctypes.cast(out, ctypes.c_void_p)
    assert lib.evo_dense_launches(0, 0, 0, 100, 256, 64, None) == -1 and lib.evo_dense_launches(0, 0, 0, 100, 250, 64, p) == -1
    assert lib.evo_dense_launches(0, 0, 1, 100, 256, 64, p) == -1 and lib.evo_dense_launches(1, 0, 1, 256, 256, 64, p) == -1


@pytest.mark.parametrize("mode,M,N,K,tile,slots", [(0, 223, 12288, 1024, 128, 0), (0, 224, 12288, 1024, 128, 6), (0, 224, 12288, 960, 128, 0), (1, 80, 22016, 4096, 96, 8),
                                                   (1, 79, 22016, 4096, 96, 0), (1, 96, 20992, 4032, 96, 0), (1, 161, 22016, 4096, 192, 5), (2, 161, 22016, 4096, 192, 5),
                                                   (1, 149, 22016, 4096, 192, 0), (1, 161, 21760, 960, 192, 0)])
def test_which_loop(mode, M, N, K, tile, slots):
    assert [(p["tile_rows"], p["slots"]) for p in all_launches(mode, False, False, M, N, K)] == [(tile, slots)]


def test_the_tile_hangs_on_the_size_and_not_on_one_width():
    """No width of K where tiles change all at once: neighbouring ones take the same launches at 98.5 of 100 sizes."""
    for mode in (0, 1):
        for K in (2112, 4096, 8192, 11008, 16320, 16384):
            other = total = 0
            for N in range(2048, 13000, 512):
                for M in range(256, 6000, 91):
                    total += 1
                    other += [tuple(p[k] for k in KEYS) for p in launches(mode, False, M, N, K)] != [tuple(p[k] for k in KEYS) for p in launches(mode, False, M, N, K - 64)]
            assert other <= 0.015 * total, (mode, K, other, total)
