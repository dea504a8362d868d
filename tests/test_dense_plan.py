"""The launches of a dense layer (csrc/gemm_tile.hip tile_plan, on the host: 256 CUs where there is no GPU): rows taken once each, statistics inside their strip."""
import ctypes

import pytest

from evo_amd import ops as evo_ops

KEYS = ("first", "rows", "tile_rows", "tile_cols", "parts", "persistent", "stat_end")


def launches(mode, stats, M, N, K):
    out = (ctypes.c_int64 * 14)()
    n = evo_ops.load_library().evo_dense_plan(mode, int(stats), M, N, K, ctypes.cast(out, ctypes.c_void_p))
    assert n in (1, 2), n
    return [dict(zip(KEYS, out[7 * i:7 * i + 7])) for i in range(n)]


# (widths of the dense layers that write the residual stream, and others whose plans end in tiles that overhang the statistic's last rows)
@pytest.mark.parametrize("N,K", [(4096, 4096), (4096, 11008), (4096, 10944), (2048, 2048), (1024, 1024), (5120, 5120), (768, 768)])
def test_statistics_stay_in_their_strip(N, K):
    overhang = 0
    for M in range(65, 12000):
        ld, end = (M + 255) // 256 * 256, 0
        for p in launches(0, True, M, N, K):
            assert p["first"] == end and p["rows"] > 0
            end += p["rows"]
            assert end <= p["stat_end"] <= ld, (M, p)             # every row's, and nothing of the next strip
            overhang += p["first"] + -(-p["rows"] // p["tile_rows"]) * p["tile_rows"] > ld
        assert end == M
    assert overhang > 0 or N == 768


def test_null_and_shapes():
    lib = evo_ops.load_library()
    out = (ctypes.c_int64 * 14)()
    assert lib.evo_dense_plan(0, 0, 100, 256, 64, None) == -1
    assert lib.evo_dense_plan(0, 0, 100, 250, 64, ctypes.cast(out, ctypes.c_void_p)) == -1
    assert lib.evo_dense_plan(3, 0, 100, 256, 64, ctypes.cast(out, ctypes.c_void_p)) == -1


def test_segments_for_a_number_of_waves():
    """From 1,024 positions (32 heads) on: the largest segment that leaves the waves asked for, 4,096 of them by default."""
    for B, T, H in ((1, 1024, 32), (8, 8193, 32), (1, 131072, 32), (3, 5000, 16)):
        for waves in (256, 4096, 65536):
            c = evo_ops.pick_segment_length(B, T, H, target_waves=waves)
            assert c in (64, 128, 256, 512, 1024)
            assert c == 64 or B * H * -(-T // c) >= waves
            assert c == 1024 or B * H * -(-T // (2 * c)) < waves
        assert evo_ops.pick_segment_length(B, T, H) == evo_ops.pick_segment_length(B, T, H, 4096)


def test_segments_of_recurrent_mixers():
    """Whole chunks, at least four; uncut where sequences and heads fill the chip; one long sequence in as many segments as there are CUs for it."""
    from evo_amd.mixer_ops import MixerOps
    plan = MixerOps.lightning_segment
    for lens in ((1,), (64,), (257,), (500,), (8190,), (131072,), (300, 5000), (1000, 2000, 3000), (4000, 4000), (1,) * 100, (1459, 1667, 1875, 2084, 2292, 2500)):
        for columns in (1, 8, 32, 64):
            for seg in (plan(lens, columns, 128 * 128), MixerOps.rglru_segment(lens, columns)):
                assert seg % 64 == 0 and seg >= 256 and (seg == 256 or seg < max(lens) + 64)
    assert plan((1459, 1667, 1875, 2084, 2292, 2500), 32, 16384) >= 2500
    assert plan((1000,) * 8, 32, 16384) >= 1000
    assert plan((4000, 4000), 32, 16384) == 1024 and plan((8190,), 32, 16384) == 1024
    plan = MixerOps.rglru_segment
    assert plan((1459, 1667, 1875, 2084, 2292, 2500), 32) >= 2500 and plan((500,), 32) == 512 and plan((8190,), 32) == 1024 and plan((1000, 2000, 4000), 32) == 1024


@pytest.mark.parametrize("N", [96, 4096, 4097, 4098, 7168, 7169, 7170, 7680, 7681, 7682, 8192, 12289, 22016, 24577, 6291456, 6291458, 6488064, 7000000, 9999998, 200000000, 2147483630])
@pytest.mark.parametrize("K", [128, 1920, 2048, 3968, 4096, 22016])
@pytest.mark.parametrize("gated", [0, 1])
def test_columns_of_weight_streaming_workgroups(N, K, gated):
    """Every column belongs to one workgroup, which has room for all of its own: floor(block cols / workgroups) up to the largest layer that is accepted, where block x
    columns has more than 32 bits.  The two halves of [W1; W2] have their borders where the gated launch has them.  A workgroup per CU for 4,097 to 7,168 columns from K = 2,048
    on and to 7,680 from 4,096 on; below, one for every 32 columns."""
    lib, out, half = evo_ops.load_library(), (ctypes.c_int64 * 4)(), (ctypes.c_int64 * 4)()
    share = lib.evo_linear_ring_share
    if gated and N % 2:
        assert share(N, K, 1, 0, ctypes.cast(out, ctypes.c_void_p)) == -1
        return
    cols = N // 2 if gated else N
    assert share(N, K, gated, 0, ctypes.cast(out, ctypes.c_void_p)) == 0 and out[1] == 0
    groups, room = out[0], out[3]
    if N <= 8192:
        assert groups == (256 if 4096 < N <= 7168 and K >= 2048 or 7168 < N <= 7680 and K >= 4096 else -(-N // 32))
    blocks = range(groups) if groups <= 120000 else sorted({0, 1, 65535, 65536, 65537, groups - 2, groups - 1} | {i * 999983 % groups for i in range(20000)})
    for b in blocks:
        assert share(N, K, gated, b, ctypes.cast(out, ctypes.c_void_p)) == 0
        assert out[0] == groups and out[1] == b * cols // groups and out[2] == (b + 1) * cols // groups and 0 < out[2] - out[1] <= room
        if gated and b % 2 == 0:
            assert share(N, K, 0, b // 2, ctypes.cast(half, ctypes.c_void_p)) == 0 and half[1] == out[1]
    assert out[2] == cols
    assert share(N, K, gated, groups, ctypes.cast(out, ctypes.c_void_p)) == -1
    assert share(N, K + 64, gated, 0, ctypes.cast(out, ctypes.c_void_p)) == share(N, 0, gated, 0, ctypes.cast(out, ctypes.c_void_p)) == -1


def test_workspace_of_segments():
    """Slots of cut sequences don't meet and stay inside the workspace, whose size follows the rows: one long prompt among many short ones asks for its own segments only."""
    import random
    from evo_amd.mixer_ops import MixerOps
    rng = random.Random(1)
    cases = [([100] * 200 + [32000], 1280), ([32000] + [50] * 400, 1280), ([0, 64, 0, 65, 128, 129], 64), ([64] * 9, 64), ([65] * 9, 64)]
    for _ in range(300):
        seg = 64 * rng.randint(1, 30)
        cases.append(([rng.choice((0, 1, seg - 1, seg, seg + 1, 3 * seg, rng.randint(0, 5 * seg))) for _ in range(rng.randint(1, 40))], seg))
    for lens, seg in cases:
        slots, at, end = MixerOps.segment_slots(len(lens), sum(lens), seg), 0, 0
        for b, n in enumerate(lens):
            if n > seg:                                           # csrc/mixers_common.h segment_slot
                first = at // seg + min(b, at // seg)
                assert first >= end
                end = first + -(-n // seg)
            at += n
        assert end <= slots <= 2 * (sum(lens) // seg)
    for many in ([100] * 200, [50] * 400):
        for lens in (many + [32000], [32000] + many):
            seg = MixerOps.lightning_segment(tuple(sorted(lens)), 32, 128 * 128)
            assert MixerOps.segment_slots(len(lens), sum(lens), seg) * 32 * 128 * 128 * 4 < 256 << 20
            seg = MixerOps.rglru_segment(tuple(sorted(lens)), 32)
            assert MixerOps.segment_slots(len(lens), sum(lens), seg) * 2 * 4096 * 4 < 16 << 20


def test_long_prompts_of_few_heads_fill_the_chip():
    """As many segments as CUs where the heads are few, and none too many where they pay nothing: several rounds of wide blocks against one."""
    from evo_amd.mixer_ops import MixerOps
    for columns in (1, 2, 4, 8, 32):
        for n in (32000, 131072):
            for seg in (MixerOps.lightning_segment((n,), columns, 128 * 128), MixerOps.rglru_segment((n,), columns)):
                assert 100 <= -(-n // seg) * columns <= 256
    six = (1459, 1667, 1875, 2084, 2292, 2500)
    assert MixerOps.rglru_segment(six, 20) == 1280 and MixerOps.rglru_segment(six, 16, small=True) <= 512
    assert MixerOps.lightning_segment(six, 32, 64 * 64) <= 768 and MixerOps.lightning_segment(six, 64, 64 * 128) >= 2500


def test_decode_attention_in_one_launch_where_caches_are_short():
    """A workgroup per key head walks its whole cache from 256 of them on, below that on short caches only: parts share a long sequence among short ones."""
    import types
    import torch
    from evo_amd.mixer_ops import MixerOps
    ops, t = types.SimpleNamespace(mixer_mfma=True), torch.zeros(1, 1, 64, dtype=torch.bfloat16)

    def whole(groups, ring, maps, dim, dv):
        return MixerOps.heads_whole_ok(ops, groups, ring, 1, maps, dim, dv, t[0], t)
    for maps, dim, dv, few, more in ((2, 128, 256, 512, 800), (1, 128, 128, 1028, 1536), (1, 64, 64, 1536, 2048)):
        assert whole(256, 1 << 20, maps, dim, dv) and not whole(79, 64, maps, dim, dv)
        for groups, ring in ((80, few), (159, few), (160, more), (255, more)):
            assert whole(groups, ring, maps, dim, dv) and not whole(groups, 2 * ring, maps, dim, dv)


def test_short_rows_by_their_width():
    """The Hyena operator in one launch: up to 4,096 channels as measured there, less of wider layers, whose rows take more rounds of workgroups; never from 1,024 positions on."""
    import torch
    p = torch.zeros(8)

    def short(B, T, D):
        return evo_ops.HipOps._hyena_short_ok(B, T, torch.empty(B, T, 3 * D, dtype=torch.bfloat16, device="meta"), None, p, p)
    for D in (128, 1024, 4096):
        assert short(1, 5, D) and short(1, 1023, D) and short(12, 41, D) and short(6, 161, D) and short(8, 90, D)
        assert not short(1, 1024, D) and not short(2, 512, D) and not short(32, 41, D) and not short(18, 5, D)
    assert short(1, 500, 8192) and short(2, 161, 8192) and not short(1, 1000, 8192) and not short(12, 41, 8192) and not short(2, 500, 8192)


def latent_forms(B, H, R, dv, n_split, prep):
    out = (ctypes.c_int64 * 5)()
    assert evo_ops.load_library().evo_latent_forms(B, H, R, dv, n_split, prep, ctypes.cast(out, ctypes.c_void_p)) == 0
    return tuple(out)


@pytest.mark.parametrize("B,H,R,dv,absorb,with_prep,up", [
    (1, 32, 512, 128, (1, 2), (1, 2), (2, 32)), (2, 32, 512, 128, (2, 2), (2, 2), (2, 32)), (8, 32, 512, 128, (4, 2), (4, 2), (2, 64)), (16, 32, 512, 128, (4, 4), (4, 4), (2, 128)),
    (32, 32, 512, 128, (4, 8), (4, 4), (4, 128)), (16, 64, 512, 128, (4, 8), (4, 4), (4, 128)), (7, 32, 512, 100, (4, 2), (4, 2), (2, 64)), (100, 128, 256, 64, (4, 8), (4, 4), (16, 128)),
    (5, 3, 40, 30, (4, 2), (4, 2), (2, 32)), (5, 3, 41, 30, (4, 1), (4, 1), (2, 32)), (33, 8, 512, 256, (4, 2), (4, 2), (4, 128))])
def test_forms_of_the_latent_maps(B, H, R, dv, absorb, with_prep, up):
    """Columns of the query side are halved while fewer than 256 workgroups take them, and are 256 at most beside the preparation; value rows while 256 workgroups are not exceeded."""
    assert latent_forms(B, H, R, dv, 16, 0) == absorb + up + (16,) and latent_forms(B, H, R, dv, 16, 1) == with_prep + up + (16,)


def test_preparation_in_the_query_sides_launch_where_it_is_ahead():
    import torch
    from evo_amd.mixer_ops import MixerOps

    def fits(B, heads, R, dn=128, dr=64):
        width = heads * (dn + dr) + R + dr
        qd, w = torch.empty(B, width, dtype=torch.bfloat16, device="meta"), torch.empty(R, dtype=torch.bfloat16, device="meta")
        return MixerOps.latent_prep_fits(qd, torch.empty(B, 64, R + dr, dtype=torch.bfloat16, device="meta"), w, torch.empty(dr // 2, device="meta"), heads, dn, dr, R)
    for B, heads, R in ((1, 32, 512), (32, 32, 512), (16, 64, 512), (64, 16, 512), (8, 128, 512), (100, 128, 256), (100, 32, 128)):
        assert fits(B, heads, R)
    for B, heads, R in ((33, 32, 512), (17, 64, 512), (65, 16, 512), (64, 128, 512), (33, 32, 384)):
        assert not fits(B, heads, R)


def test_no_more_parts_in_flight_than_there_are():
    for n in range(1, 65):
        assert latent_forms(16, 32, 512, 128, n, 0)[4] == (4 if n <= 4 else 8 if n <= 8 else 16)


def tiles(M, N, K):
    p, = launches(0, False, M, N, K)
    return p["tile_rows"], p["tile_cols"], p["parts"]


@pytest.mark.parametrize("N", [5632, 5888, 6144])
def test_narrow_tiles_where_they_are_ahead(N):
    """96 x 48: not where the second row tile is nearly empty and K is small, nor where parts of a long K are ahead."""
    for K, first, last in ((2048, 112, 192), (2496, 112, 192), (2560, 97, 192), (4096, 97, 192), (4608, 97, 192), (4672, 97, 144), (5120, 97, 144)):
        for M in range(97, 193):
            assert (tiles(M, N, K) == (96, 48, 1)) == (first <= M <= last), (M, K, tiles(M, N, K))


def test_parts_for_a_norm_where_they_are_ahead():
    """Layers whose own launch is ahead of parts and their norm, and neighbours whose is not."""
    parts = evo_ops.load_library().evo_dense_parts
    for M, N, K in ((900, 4096, 5632), (780, 4096, 5632), (940, 4096, 5632), (660, 4096, 4096), (900, 3072, 3072), (136, 3072, 3072), (151, 3072, 3072),
                    (130, 4096, 4096), (138, 4096, 4096)):
        assert parts(M, N, K) == 0, (M, N, K)
    for M, N, K in ((1000, 4096, 5632), (740, 4096, 5632), (700, 4096, 5632), (600, 4096, 4096), (512, 4096, 4096), (880, 3072, 3072), (128, 3072, 3072), (123, 4096, 4096),
                    (145, 4096, 4096), (161, 4096, 4096), (181, 3072, 3584), (189, 3072, 4096), (296, 2048, 4096), (435, 1536, 3584), (161, 3584, 4096),
                    (222, 4096, 5632), (161, 4096, 11008), (90, 6144, 4096), (145, 5120, 5120)):
        assert parts(M, N, K) >= 2, (M, N, K)
