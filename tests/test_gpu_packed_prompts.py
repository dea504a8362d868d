"""GPU: unequal StripedHyena prompts in one pass (StripedHyena._prefill_packed) against the same prompts one by one, and the decode steps behind both.
Tolerance: the two differ in the dense layers' tiles and, from 1,024 rows on, in where the norms' weights are rounded -- two bf16 evaluations of the same
model, each within 2e-2 of fp64 on these four layers (tests/test_gpu_pool.py); a mixed-up row, position or state is off by its whole norm."""
import pytest
import torch

from test_gpu_model import DEV, SMALL4, build

pytestmark = pytest.mark.gpu
WIDE = dict(vocab_size=512, hidden_size=4096, num_layers=4, attn_layer_idxs=[1], num_attention_heads=32)


def prompts_of(lens):
    g = torch.Generator().manual_seed(sum(lens))
    letters = torch.tensor(list(b"ACGT"))
    return [letters[torch.randint(0, 4, (n,), generator=g)].to(DEV) for n in lens]


# lengths at the edges of 64-row places, 512-step tiles, the 32-token limit of the matrix-core operator and the 128-row attention kernel; few and many rows
@pytest.mark.parametrize("dims,lens", [("toy", [33, 64, 65, 5, 127, 32, 31]), ("toy", [512, 513, 129, 40, 300]), ("wide", [40, 64, 70]),
                                       ("wide", [511, 512, 513, 33, 8, 1025, 128])])
def test_packed_prompts_are_the_prompts_alone(dims, lens):
    from evo_amd.pool import DecodePool
    _, _, m = build(dict(SMALL4 if dims == "toy" else WIDE, use_interpolated_rotary_pos_emb=True, rotary_emb_scaling_factor=16))
    prompts = prompts_of(lens)
    want = [sorted({0, n // 2, n - 1}) for n in lens]
    assert max(len(g) for g in m._prompt_groups(lens)) > 1
    nxt = prompts_of([4] * len(lens))
    packed, alone = DecodePool(m, None, n_slots=len(lens)), DecodePool(m, None, n_slots=len(lens))
    slots, lg = packed.admit(prompts, want, reserve=8)
    first, lg1 = [], []
    for p, w in zip(prompts, want):
        s, l = alone.admit([p], [w], reserve=8)
        first += s
        lg1 += l

    def close(a, b, what):
        assert ((a - b).norm() / b.norm()).item() < 3e-2, what
    for n, (a, b) in enumerate(zip(lg, lg1)):
        for r in range(a.shape[0]):
            close(a[r], b[r], (lens[n], want[n][r]))
    for b, n in enumerate(lens):
        close(packed.ipd["mha"].key_value_memory_dict[1][slots[b], :n].float(), alone.ipd["mha"].key_value_memory_dict[1][first[b], :n].float(), ("kv", n))
        for i in m.hyena_layer_idxs:
            close(torch.view_as_real(packed.ipd["hyena"].state_dict[i][slots[b]]), torch.view_as_real(alone.ipd["hyena"].state_dict[i][first[b]]), ("state", i, n))
            close(packed.ipd["hyena"].fir_state_dict[i][slots[b]].float(), alone.ipd["hyena"].fir_state_dict[i][first[b]].float(), ("fir", i, n))
    for k in range(4):
        a = packed.advance({s: int(t[k]) for s, t in zip(slots, nxt)})
        b = alone.advance({s: int(t[k]) for s, t in zip(first, nxt)})
        for i, (s, f) in enumerate(zip(slots, first)):
            close(a[s], b[f], ("step", k, lens[i]))


def test_caches_take_the_prompts_own_lengths():
    """Short prompts beside a long one: the keys and values that a pass keeps are those of its tokens."""
    from evo_amd.pool import DecodePool
    _, _, m = build(dict(SMALL4))
    lens = [33, 2000] + [40] * 30
    assert len(m._prompt_groups(lens)) == 1
    got = DecodePool(m, None, n_slots=2).prefill(prompts_of(lens))
    kept = {}
    for (_, ipd, row), n in zip(got, lens):
        kv = ipd["mha"].key_value_memory_dict[1]
        assert kv.shape[1] >= n and row < kv.shape[0]
        kept[kv.untyped_storage().data_ptr()] = kv.untyped_storage().nbytes()
    assert sum(kept.values()) == sum(lens) * 2 * m.hidden_size * 2


def test_places_from_the_end_and_places_that_are_not_there():
    _, _, m = build(dict(SMALL4))
    lens = [40, 65, 33]
    prompts = prompts_of(lens)
    with torch.inference_mode():
        for group in (prompts, prompts[:1]):                     # packed, alone
            a = m.prefill_rows(group, [[-1, -len(p), 5] for p in group])
            b = m.prefill_rows(group, [[len(p) - 1, 0, 5] for p in group])
            for x, y in zip(a, b):
                assert torch.equal(x[0], y[0])
            for bad in (len(group[0]), -len(group[0]) - 1):
                with pytest.raises(IndexError):
                    m.prefill_rows(group, [[bad]] + [[0]] * (len(group) - 1))


@pytest.mark.parametrize("dims", ["toy", "wide"])
@pytest.mark.parametrize("n", [1024, 2304, 3584])
def test_whole_row_tiles_have_the_same_bits_alone_and_packed(dims, n):
    """A prompt of 1,024 tokens and more, a multiple of 256: its keys, values and states are the same bits alone and beside others, either side of 3,500 keys."""
    _, _, m = build(dict(SMALL4 if dims == "toy" else WIDE))
    p = prompts_of([n, 300, 700, 1200])
    with torch.inference_mode():
        _, alone, row = m.prefill_rows([p[0]])[0]
        for at, group in ((0, [p[0], p[1]]), (1, [p[2], p[0], p[3]])):
            assert len(m._prompt_groups([q.numel() for q in group])) == 1
            _, ipd, r = m.prefill_rows(group)[at]
            assert torch.equal(ipd["mha"].key_value_memory_dict[1][r, :n], alone["mha"].key_value_memory_dict[1][row, :n])
            for i in m.hyena_layer_idxs:
                a, b = (torch.view_as_real(d["hyena"].state_dict[i][k]) for d, k in ((ipd, r), (alone, row)))
                assert torch.equal(a.reshape(b.shape), b)
